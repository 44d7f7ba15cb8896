// spmv.hip -- ABHSF SpMV / SpMM kernels for gfx950 (wave64).
//
// One wavefront owns one strip (block row of s rows) and accumulates its
// s x R output tile in LDS; the four scheme groups of the strip are walked in
// turn (COO, CSR, bitmap, dense), each with a decode specialised to its layout.
// One right-hand side:
//   COO / CSR  entry-parallel in storage order, 64 consecutive entries per
//              load; an entry's block (COO) or block row (CSR) is the number of
//              segment ends before it in a bit mask in LDS;
//   bitmap     a lane owns consecutive positions and walks their set bits;
//   dense      16- and 32-row blocks in 1 KB wave steps, else as bitmap.
// Several right-hand sides: COO and bitmap windows of 64 entries decoded into
// LDS (block by binary search over the chunk's prefix sums), CSR rows by lane,
// dense blocks on the FP64 matrix cores where the tile is wide enough.
// Products of the same output row are summed in registers and DPP where rows
// are known to be contiguous (bitmap, dense) and with LDS atomic adds where
// they are not.
//
// Reference semantics: y[lrow] += v * x[bcol*s + lcol] per scheme
// (spmv/orig/88.cpp:214-235 COO, 88_bitmap.cpp:183-207 bitmap, 88.cpp:587-604
// dense); the whole-matrix call is y = alpha*A*x + beta*y, which with
// alpha = beta = 1 is the accumulating csr_matrix::spmv of
// spmv/unified/spmv.cpp:140-159.
//
// COMP (FP32 value storage): every product is split exactly with an FMA
// (TwoProduct) and every LDS accumulation is made error-free with TwoSum: the
// atomic returns the old value a, so the rounding error of fl(a + p) is
// recovered exactly and added to a second accumulator (Ogita, Rump, Oishi,
// "Accurate sum and dot product", SIAM J. Sci. Comput. 26(6), 2005, Dot2).
#include "spmv.hpp"

#include <algorithm>
#include <type_traits>

namespace abhsf {
namespace {

// The single-RHS kernels read the matrix descriptor through the constant
// address space, field by field where a group needs it (scalar loads), and
// each group starts from a pointer and a lane number the compiler cannot see
// through.  With the descriptor passed by value the compiler kept fields and
// lane addresses of all four groups for the whole kernel: 83 VGPRs and 57
// spilled SGPRs where the same groups now take 67 and none (FP64 values).
using MatPtr = const __attribute__((address_space(4))) DevMat *;
using BalPtr = const __attribute__((address_space(4))) Balance *;

template <typename P>
__device__ inline P opaque_s(P p)
{
    const uint64_t v = (uint64_t)p;
    uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    asm volatile("" : "+s"(lo), "+s"(hi));
    return (P)(((uint64_t)hi << 32) | lo);
}
__device__ inline int opaque_v(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// A pointer read from a descriptor, known to point to device memory (global
// instead of flat loads).
template <typename T>
__device__ inline const T *glob(const void *p)
{
    return (const T *)(const __attribute__((address_space(1))) T *)p;
}
template <typename T>
__device__ inline T *glob_rw(T *p)
{
    return (T *)(__attribute__((address_space(1))) T *)p;
}

template <typename T>
__device__ inline T ld(const void *p, uint64_t i) { return static_cast<const T *>(p)[i]; }

// x may be any double pointer (x + 1 of a caller's array included); the
// paired loads of the dense paths take it as double2 only when it is 16-byte
// aligned.
__device__ inline bool x_aligned16(const double *x) { return (reinterpret_cast<uintptr_t>(x) & 15u) == 0; }

struct Acc {
    double *hi;  // [s * R]
    double *lo;  // [s * R] (COMP only)
};

// Atomic accumulate of p into acc slot i.
template <bool COMP>
__device__ inline void acc_atomic(const Acc &a, uint32_t i, double p, double perr)
{
    if constexpr (COMP) {
        double old = atomicAdd(&a.hi[i], p);
        double s, e;
        two_sum(old, p, s, e);
        atomicAdd(&a.lo[i], e + perr);
    } else {
        atomicAdd(&a.hi[i], p);
    }
}

// Product v*x, with its exact rounding error when COMP.
template <bool COMP>
__device__ inline double prod(double v, double x, double &err)
{
    double p = v * x;
    if constexpr (COMP) err = __builtin_fma(v, x, -p); else err = 0.0;
    return p;
}

// ===========================================================================
// Single right-hand side (SpMV).
// ===========================================================================

// Accumulate p (with product error pe) into a lane-private compensated pair.
template <bool COMP>
__device__ inline void acc_add(double &hi, double &lo, double v, double xv)
{
    if constexpr (COMP) {
        double pe;
        const double p = prod<true>(v, xv, pe);
        double s, e;
        two_sum(hi, p, s, e);
        hi = s;
        lo += e + pe;
    } else {
        hi = __builtin_fma(v, xv, hi);
    }
}

// Sum (hi, lo) over aligned groups of P lanes (P = 2 or 4).
template <bool COMP, int P>
__device__ inline void group_reduce_p(double &hi, double &lo)
{
    if constexpr (!COMP) {
        hi = group_sum_dpp<P>(hi);
    } else {
        auto step = [&](auto ctrl_tag) {
            constexpr int CTRL = decltype(ctrl_tag)::value;
            const double th = dpp_f64<CTRL>(hi), tl = dpp_f64<CTRL>(lo);
            double s, e;
            two_sum(hi, th, s, e);
            hi = s;
            lo += tl + e;
        };
        step(std::integral_constant<int, DPP_QUAD_XOR1>{});
        if constexpr (P == 4) step(std::integral_constant<int, DPP_QUAD_XOR2>{});
    }
}

// Sum (hi, lo) over aligned groups of 2^k lanes, 1 <= k <= 4 (uniform).
template <bool COMP>
__device__ __forceinline__ void row_reduce(int k, double &hi, double &lo)
{
    auto step = [&](auto ctrl_tag) {
        constexpr int CTRL = decltype(ctrl_tag)::value;
        const double th = dpp_f64<CTRL>(hi);
        if constexpr (COMP) {
            const double tl = dpp_f64<CTRL>(lo);
            double s, e;
            two_sum(hi, th, s, e);
            hi = s;
            lo += tl + e;
        } else {
            hi += th;
        }
    };
    step(std::integral_constant<int, DPP_QUAD_XOR1>{});
    if (k > 1) step(std::integral_constant<int, DPP_QUAD_XOR2>{});
    if (k > 2) step(std::integral_constant<int, DPP_ROW_HALF_MIRROR>{});
    if (k > 3) step(std::integral_constant<int, DPP_ROW_MIRROR>{});
}

// (P = 1, 2 or 4)
template <bool COMP>
__device__ inline void group_reduce(int P, double &hi, double &lo)
{
    if (P == 2) group_reduce_p<COMP, 2>(hi, lo);
    else if (P == 4) group_reduce_p<COMP, 4>(hi, lo);
}

// LDS of one wave besides its accumulator: a chunk's segments (COO blocks, or
// the rows of CSR blocks that hold entries) and the mask of their ends.
constexpr int kSegs = 4 * kWave;   // segments per chunk, four per lane
constexpr int kMaskEnts = 2048;    // entries one mask covers
// Any four COO blocks fit a mask: the cost model gives a block to COO only up
// to 2s entries (2 lg(s) z + 2 lg(s) <= lg(s) z + (s + 1) 2 lg(s)).
static_assert(4 * 2 * 256 <= kMaskEnts, "four COO blocks per mask");

struct WaveLds {
    uint32_t bc[kSegs];              // first column of every segment's block
    uint64_t ends[kMaskEnts / 64];   // bit t: entry t is its segment's last
    uint16_t to[kSegs];              // first accumulator row of the block's strip; CSR: the row
};

// Values of segments' blocks [cb, cb + nbk) of a per-block array, four
// consecutive blocks per lane (0 past the end): one 4- or 8- or 16-byte load
// per lane, single ones in the last lane.
template <typename T>
__device__ __forceinline__ void load4(const T *__restrict__ a, uint32_t cb, uint32_t nbk, int lane, uint32_t (&v)[4])
{
    const uint32_t j = 4u * (uint32_t)lane;
    const T *__restrict__ p = a + cb + j;
    T w[4] = {0, 0, 0, 0};
    if (j + 4u <= nbk) {
        __builtin_memcpy(w, p, sizeof(w));
    } else {
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (j + (uint32_t)i < nbk) w[i] = p[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = (uint32_t)w[i];
}

// How an entry's row and column follow from its index and its segment.
enum SegMode { SEG_COO, SEG_STRIPS, SEG_CSR };  // (one strip, several, CSR rows with FP32 values)

// Windows of 64 consecutive entries from vp / ip on (values and in-block
// indices: COO (lrow << k) | lcol, CSR lcol), T <= kMaskEnts entries in nseg
// segments whose ends are marked in L.ends; `before` segments end before the
// first one.  Values and indices are read 64 consecutive ones per load, U
// windows in flight; an entry's segment is the number of end bits before it
// (mbcnt over the window's mask word plus a running count).
template <typename VT, typename IT, bool COMP, int MODE, int U>
__device__ __forceinline__ void seg_windows(const VT *__restrict__ vp, const IT *__restrict__ ip, uint32_t T,
                                            uint32_t nseg, uint32_t before, int k, const double *__restrict__ x,
                                            const Acc &acc, const WaveLds &L, int lane_)
{
    const int lane = opaque_v(lane_);  // its addresses are not kept outside
    const uint32_t smask = (1u << k) - 1u;
    // W windows from entry q on; TAIL: the last of them is not full (its lanes
    // past the last entry read that one again and add nothing)
    auto windows = [&](uint32_t q, auto w_tag, auto tail_tag) __attribute__((always_inline)) {
        constexpr int W = decltype(w_tag)::value;
        constexpr bool TAIL = decltype(tail_tag)::value;
        auto live = [&](int u) { return !(TAIL && u == W - 1) || q + (uint32_t)(u * kWave + lane) < T; };
        uint32_t id[W], r[W];
        double v[W], xv[W];
#pragma unroll
        for (int u = 0; u < W; u++) {
            uint32_t t = (uint32_t)(u * kWave + lane);
            if (TAIL && u == W - 1) t = min(t, T - 1u - q);
            id[u] = (ip + q)[t];
            v[u] = (double)(vp + q)[t];
        }
#pragma unroll
        for (int u = 0; u < W; u++) {
            const uint64_t m = L.ends[q / kWave + (uint32_t)u];
            const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
            uint32_t own = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, before));
            if (TAIL && u == W - 1) own = min(own, nseg - 1u);
            before += (uint32_t)__popc(lo) + (uint32_t)__popc(hi);
            if constexpr (MODE == SEG_CSR) {
                r[u] = L.to[own];
                xv[u] = x[L.bc[own] + id[u]];
            } else {
                r[u] = id[u] >> k;
                if constexpr (MODE == SEG_STRIPS) r[u] += (uint32_t)L.to[own];
                xv[u] = x[L.bc[own] + (id[u] & smask)];
            }
        }
        if constexpr (COMP) {
            // every returning add first, then the TwoSums and the compensation
            // adds (hi and lo receive their adds in entry order either way):
            // the returns are awaited once
            double pr[W], pe[W], old[W];
#pragma unroll
            for (int u = 0; u < W; u++) {
                pr[u] = prod<true>(v[u], xv[u], pe[u]);
                if (live(u)) old[u] = atomicAdd(&acc.hi[r[u]], pr[u]);
            }
#pragma unroll
            for (int u = 0; u < W; u++)
                if (live(u)) {
                    double sum, err;
                    two_sum(old[u], pr[u], sum, err);
                    atomicAdd(&acc.lo[r[u]], err + pe[u]);
                }
        } else {
#pragma unroll
            for (int u = 0; u < W; u++)
                if (live(u)) atomicAdd(&acc.hi[r[u]], v[u] * xv[u]);
        }
    };
    using std::integral_constant;
    uint32_t q = 0;
    // Full steps of long segments: a lane takes four consecutive entries and
    // adds runs of one row as one sum.  Entries of a row lie side by side, and
    // adds to one address are taken one lane at a time: with consecutive
    // entries in consecutive lanes block_mix n = 217 081 s = 256 tiled (32
    // consecutive entries a row) took 105 us with FP32 values, now 41 us;
    // 32-row random blocks s = 128 41 -> 25 us.  COO blocks of few entries
    // have no such runs (R-MAT scale 20 s = 256, 6 a block: 66 us, 71 this
    // way) except where the adds return (FP32 values).
    if (U == 4 && (COMP || T >= 16u * nseg)) {
#pragma unroll 1
        for (; q + (uint32_t)(4 * kWave) <= T; q += (uint32_t)(4 * kWave)) {
            VT vw[4];
            IT iw[4];
            __builtin_memcpy(vw, vp + q + 4u * (uint32_t)lane, sizeof(vw));
            __builtin_memcpy(iw, ip + q + 4u * (uint32_t)lane, sizeof(iw));
            const uint32_t nib = (uint32_t)(L.ends[q / kWave + (uint32_t)(lane >> 4)] >> (4 * (lane & 15))) & 15u;
            const uint32_t cnt = (uint32_t)__popc(nib), incl = wave_incl_scan_dpp(cnt);
            const uint32_t own0 = before + incl - cnt;
            before += (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
            uint32_t r[4];
            double xv[4], hi[4], lo[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t own = own0 + (uint32_t)__popc(nib & ((1u << i) - 1u)), id = (uint32_t)iw[i];
                if constexpr (MODE == SEG_CSR) {
                    r[i] = L.to[own];
                    xv[i] = x[L.bc[own] + id];
                } else {
                    r[i] = id >> k;
                    if constexpr (MODE == SEG_STRIPS) r[i] += (uint32_t)L.to[own];
                    xv[i] = x[L.bc[own] + (id & smask)];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                hi[i] = prod<COMP>((double)vw[i], xv[i], lo[i]);
                if (i && r[i] == r[i - 1]) {
                    if constexpr (COMP) {
                        double sum, err;
                        two_sum(hi[i - 1], hi[i], sum, err);
                        hi[i] = sum;
                        lo[i] += lo[i - 1] + err;
                    } else {
                        hi[i] += hi[i - 1];
                    }
                }
            }
            auto last = [&](int i) { return i == 3 || r[i + 1] != r[i]; };
            if constexpr (COMP) {
                // every returning add first, then the TwoSums and the
                // compensation adds: the returns are awaited once
                double old[4];
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (last(i)) old[i] = atomicAdd(&acc.hi[r[i]], hi[i]);
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (last(i)) {
                        double sum, err;
                        two_sum(old[i], hi[i], sum, err);
                        atomicAdd(&acc.lo[r[i]], err + lo[i]);
                    }
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (last(i)) atomicAdd(&acc.hi[r[i]], hi[i]);
            }
        }
    }
#pragma unroll 1
    for (; q + (uint32_t)(U * kWave) <= T; q += (uint32_t)(U * kWave))
        windows(q, integral_constant<int, U>{}, std::false_type{});
    const uint32_t left = T - q;  // uniform
    if (U > 3 && left > 3u * kWave) windows(q, integral_constant<int, 4>{}, std::true_type{});
    else if (U > 2 && left > 2u * kWave) windows(q, integral_constant<int, 3>{}, std::true_type{});
    else if (U > 1 && left > (uint32_t)kWave) windows(q, integral_constant<int, 2>{}, std::true_type{});
    else if (left) windows(q, integral_constant<int, 1>{}, std::true_type{});
}

// CSR entries of a mask (FP64 values; vp, ip, T, nseg, before as in
// seg_windows): four consecutive entries per lane, a row (segment) summed by
// fma from entry to entry.  A lane's open sum takes in the next lane's first
// one if the row ends there (not across 16 lanes), so most rows of up to eight
// entries are added once to the strip's sums.
// Every entry added by itself (seg_windows) took 1 to 6 % less time (27-point
// stencil 160^3 s = 64 250 us, here 253; s = 128 250, here 265), but rounded
// each product and let a row's small terms meet the strip's sum one by one:
// 32 % more error (rms) for the stencil at s = 32, 25 % at s = 64.
__device__ __forceinline__ void csr_sums(const double *__restrict__ vp, const uint8_t *__restrict__ ip, uint32_t T,
                                         uint32_t nseg, uint32_t before, const double *__restrict__ x, const Acc &acc,
                                         const WaveLds &L, int lane_)
{
    const int lane = opaque_v(lane_);
    // 256 entries from q on; TAIL: fewer
    auto quads = [&](uint32_t q, auto tail_tag) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail_tag)::value;
        const uint32_t t = q + 4u * (uint32_t)lane;
        double v[4], xv[4], p[4];
        uint8_t id[4];
        if constexpr (TAIL) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t j = min(t + (uint32_t)i, T - 1u);
                v[i] = vp[j];
                id[i] = ip[j];
            }
        } else {
            __builtin_memcpy(v, vp + t, sizeof(v));
            __builtin_memcpy(id, ip + t, sizeof(id));
        }
        // end bits: of the lane's entries, of the next lane's (none for the
        // last of 16 lanes), of the entry before
        const uint64_t word = L.ends[q / kWave + (uint32_t)(lane >> 4)];
        const int sh = 4 * (lane & 15);
        const uint32_t nib = (uint32_t)(word >> sh) & 15u, next = (uint32_t)(word >> sh) >> 4 & 15u;
        const bool taken = sh && nib && !((word >> ((sh - 1) & 63)) & 1ull);
        const uint32_t cnt = (uint32_t)__popc(nib), incl = wave_incl_scan_dpp(cnt);
        const uint32_t own0 = before + incl - cnt;
        before += (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        uint32_t r[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t own = own0 + (uint32_t)__popc(nib & ((1u << i) - 1u));
            if (TAIL) own = min(own, nseg - 1u);
            r[i] = L.to[own];
            xv[i] = x[L.bc[own] + (uint32_t)id[i]];
            if (TAIL && t + (uint32_t)i >= T) {
                v[i] = 0.0;
                xv[i] = 0.0;
            }
        }
        p[0] = v[0] * xv[0];
#pragma unroll
        for (int i = 1; i < 4; i++) p[i] = __builtin_fma(v[i], xv[i], (nib >> (i - 1)) & 1u ? 0.0 : p[i - 1]);
        const uint32_t last = TAIL ? (t < T ? min(T - t, 4u) - 1u : 4u) : 3u;  // (4: no entries)
        const bool open = last < 4u && !((nib >> last) & 1u);
        const double in = dpp_f64<DPP_ROW_SHL1>(nib & 1u ? p[0] : nib & 2u ? p[1] : nib & 4u ? p[2] : p[3]);
        if (open && next) p[3] += in;
        uint32_t put = taken ? nib & (nib - 1u) : nib;
        if (open) put |= 8u;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if ((put >> i) & 1u) atomicAdd(&acc.hi[r[i]], p[i]);
    };
    uint32_t q = 0;
#pragma unroll 1
    for (; q + (uint32_t)(4 * kWave) <= T; q += (uint32_t)(4 * kWave)) quads(q, std::false_type{});
    const uint32_t left = T - q;
    if (left > (uint32_t)kWave) {
        quads(q, std::true_type{});
    } else if (left) {  // one entry per lane, each added to the strip's sums
        const uint32_t t = q + min((uint32_t)lane, left - 1u);
        const double v = vp[t];
        const uint32_t id = ip[t];
        const uint64_t m = L.ends[q / kWave];
        const uint32_t own = min((uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, before)),
                                 nseg - 1u);
        const uint32_t r = L.to[own];
        const double xv = x[L.bc[own] + id];
        if ((uint32_t)lane < left) atomicAdd(&acc.hi[r], v * xv);
    }
}

// CSR group, blocks [b0, b1) whose first value is at offset e.  Chunks of 256
// block rows (256 / s blocks), four consecutive rows of a block per lane: the
// rows that hold entries are the chunk's segments (their number in L.to, the
// block's first column in L.bc), the row pointers give their ends, and the
// entries are taken in storage order (csr_sums; FP32 values as COO blocks).
// Bound: memory latency.  When the lane of a row walked the row's entries by
// itself, one load of 3-entry rows touched 12 lines instead of 4 and waited
// for the row pointers, and a long row held up the wave for its whole length
// (R-MAT scale 20 s = 256 tiled, 10 % of the entries in CSR blocks, 124 -> 69
// us; block_mix n = 2^22 s = 128 tiled 983 -> 654 us).
// A group of T > 1 strips from I0 on: strip I0 + t has the accumulator rows
// from t << k on.
template <typename VT, typename BT, typename RT, bool COMP>
__device__ __forceinline__ void csr_r1(MatPtr A_, uint32_t b0, uint32_t b1, uint32_t e, const double *__restrict__ x,
                                       const Acc &acc, WaveLds &L, int lane_, int64_t I0 = 0, int T_ = 1)
{
    if (b0 >= b1) return;
    const MatPtr A = opaque_s(A_);
    const int lane = opaque_v(lane_);
    const int k = A->k;
    const VT *__restrict__ val = glob<VT>(A->val[CSR]);
    const uint8_t *__restrict__ ccol = glob<uint8_t>(A->csr_col);
    const RT *__restrict__ rowptr = glob<RT>(A->csr_rowptr);
    const BT *__restrict__ bcol = glob<BT>(A->bcol[CSR]);
    uint32_t *ends32 = reinterpret_cast<uint32_t *>(L.ends);
    const uint32_t nb = (uint32_t)kSegs >> k;  // blocks per chunk (the cost model has no CSR blocks below s = 16)
    const uint32_t j = (4u * (uint32_t)lane) >> k, r0 = (4u * (uint32_t)lane) & ((1u << k) - 1u);
#pragma unroll 1
    for (uint32_t cb = b0; cb < b1; cb += nb) {
        uint32_t a[5] = {0, 0, 0, 0, 0}, bc = 0, row = r0;
        for (int t = 1; t < T_; t++)  // the block's strip
            if (cb + j >= glob<uint32_t>(A->sptr[CSR])[I0 + t]) row = r0 + ((uint32_t)t << k);
        if (cb + j < b1) {
            const RT *__restrict__ rp = rowptr + ((uint64_t)(cb + j) * (uint64_t)((1u << k) + 1u) + r0);
            RT w[4];
            __builtin_memcpy(w, rp, sizeof(w));
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = (uint32_t)w[i];
            a[4] = (uint32_t)rp[4];
            bc = (uint32_t)bcol[cb + j] << k;
        }
        // prefix sums of the entries (low half) and of the rows that hold some
        uint32_t rows = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) rows += a[i + 1] != a[i];
        const uint32_t mine = (a[4] - a[0]) | (rows << 16);
        const uint32_t incl = wave_incl_scan_dpp(mine);
        const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        const uint32_t T = tot & 0xFFFFu, nseg = tot >> 16;
        // chunk positions of the rows' last entries, two per register (the
        // cost model keeps a chunk's CSR blocks below 2^13 entries in all;
        // none: 0xFFFF)
        const uint32_t p0 = ((incl - mine) & 0xFFFFu) - a[0];
        uint32_t o = (incl - mine) >> 16, last[2] = {~0u, ~0u};
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (a[i + 1] != a[i]) {
                L.bc[o] = bc;
                L.to[o] = (uint16_t)(row + (uint32_t)i);
                o++;
                last[i / 2] ^= (0xFFFFu ^ (p0 + a[i + 1] - 1u)) << (16 * (i & 1));
            }
#pragma unroll 1
        for (uint32_t w = 0; w < T; w += (uint32_t)kMaskEnts) {
            const uint32_t Tw = min(T - w, (uint32_t)kMaskEnts);
            ends32[lane] = 0u;
            wave_sync();
            uint32_t before = 0;  // rows that end before entry w
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t t = (last[i / 2] >> (16 * (i & 1))) & 0xFFFFu;
                before += t < w;
                if (t - w < Tw) atomicOr(&ends32[(t - w) >> 5], 1u << ((t - w) & 31u));
            }
            if (w) before = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan_dpp(before), kWave - 1);
            wave_sync();
            if constexpr (COMP)
                seg_windows<VT, uint8_t, COMP, SEG_CSR, 4>(val + (e + w), ccol + (e + w), Tw, nseg, before, k, x, acc,
                                                           L, lane);
            else
                csr_sums(val + (e + w), ccol + (e + w), Tw, nseg, before, x, acc, L, lane);
            wave_sync();
        }
        e += T;
    }
}

// Group of T consecutive strips from I0 on, scheme SC: the first block of strip
// I0 + lane, ~0 where the strip has none (lane < T <= 64).
template <int SC>
__device__ __forceinline__ uint32_t group_first(MatPtr A, int64_t I0, int T, int lane)
{
    uint32_t first = ~0u;
    if (lane < T) {
        const uint32_t *sp = glob<uint32_t>(A->sptr[SC]) + I0 + lane;
        const uint32_t f0 = sp[0], f1 = sp[1];
        if (f1 > f0) first = f0;
    }
    return first;
}

// First accumulator rows (t << k) of the blocks [cb, cb + nbk) of a group, four
// consecutive blocks per lane, into L.to: a block's strip t is the last one
// that starts at or before it, so every strip leaves its rows at its first
// block and a running maximum spreads them.
__device__ __forceinline__ void group_rows(uint32_t first, uint32_t cb, uint32_t nbk, int k, WaveLds &L, int lane)
{
    *reinterpret_cast<uint2 *>(&L.to[4 * lane]) = make_uint2(0u, 0u);
    wave_sync();
    if (first > cb && first < cb + nbk) L.to[first - cb] = (uint16_t)(lane << k);
    wave_sync();
    const uint32_t t0 = (uint32_t)(63 - __clzll(__ballot(first <= cb))) << k;  // block cb's
    const uint2 w = *reinterpret_cast<const uint2 *>(&L.to[4 * lane]);
    uint32_t to[4];
    to[0] = w.x & 0xFFFFu;
    to[1] = max(to[0], w.x >> 16);
    to[2] = max(to[1], w.y & 0xFFFFu);
    to[3] = max(to[2], w.y >> 16);
    const uint32_t up = wave_incl_max_dpp(max(to[3], t0));
    const uint32_t left = (uint32_t)__shfl_up((int)up, 1, kWave);  // (every lane takes part)
    const uint32_t before = lane ? left : t0;
#pragma unroll
    for (int i = 0; i < 4; i++) to[i] = max(to[i], before);
    *reinterpret_cast<uint2 *>(&L.to[4 * lane]) = make_uint2(to[0] | (to[1] << 16), to[2] | (to[3] << 16));
}

// COO group, blocks [b0, b1) with first value at offset e.  Chunks of up to
// 256 blocks (four per lane, one prefix sum) and 2048 entries; a block is a
// segment: it sets the bit of its last entry in the LDS mask and leaves its
// first column in LDS.  The chunk's entries are taken in storage order, at
// addresses known before the block metadata arrive.  A block's z1 holds z - 1
// in its low A.zb bits and, in a tile, the block's strip t within the tile
// above them: the row is (t << k) + lrow.  In a group of consecutive strips
// the blocks lie in strip order (group_rows).
// Bound: memory latency and the x gathers.  Before, a binary search of the
// prefix sums located every entry beyond a block's first two, which the
// block's lane took by itself: 62 VALU instructions per 64 entries (28 now)
// and loads that waited for the metadata.  Together with entries in storage
// order for CSR blocks: 27-point stencil 160^3 s = 64 394 -> 249 us (4.7 TB/s),
// R-MAT scale 22 s = 256 tiled 470 -> 356 us.
enum CooMode { COO_STRIP, COO_TILE, COO_GROUP };

template <typename VT, typename BT, typename IT, bool COMP, int MODE = COO_STRIP>
__device__ __forceinline__ void coo_r1(MatPtr A_, uint32_t b0, uint32_t b1, uint32_t e, const double *__restrict__ x,
                                       const Acc &acc, WaveLds &L, int lane_, int windows = 4, int64_t I0 = 0,
                                       int T_ = 1)
{
    if (b0 >= b1) return;
    constexpr bool TILE = MODE == COO_TILE;
    const MatPtr A = opaque_s(A_);
    const int lane = opaque_v(lane_);
    const int k = A->k, zb = TILE ? A->zb : 16;
    const uint32_t zmask = (1u << zb) - 1u;
    const VT *__restrict__ val = glob<VT>(A->val[COO]);
    const IT *__restrict__ idx = glob<IT>(A->coo_idx);
    const uint16_t *__restrict__ z1 = glob<uint16_t>(A->z1[COO]);
    const BT *__restrict__ bcol = glob<BT>(A->bcol[COO]);
    uint32_t *ends32 = reinterpret_cast<uint32_t *>(L.ends);
    uint32_t cb = b0, first = ~0u;
    if constexpr (MODE == COO_GROUP) first = group_first<COO>(A, I0, T_, lane);
#pragma unroll 1
    while (cb < b1) {
        uint32_t nbk = min<uint32_t>(kSegs, b1 - cb);
        uint32_t z[4], bc[4];
        load4(z1, cb, nbk, lane, z);
        load4(bcol, cb, nbk, lane, bc);
        uint32_t to[4], zs = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (TILE) {
                to[i] = (z[i] >> zb) << k;
                z[i] &= zmask;
            }
            z[i] = 4u * (uint32_t)lane + (uint32_t)i < nbk ? z[i] + 1u : 0u;
            zs += z[i];
            bc[i] <<= k;
        }
        const uint32_t incl = wave_incl_scan_dpp(zs);
        uint32_t T = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        bool mine = true;
        if (T > (uint32_t)kMaskEnts) {  // uniform: take the lanes whose blocks fit
            mine = incl <= (uint32_t)kMaskEnts;
            const int nl = __popcll(__ballot(mine));
            T = (uint32_t)__builtin_amdgcn_readlane((int)incl, nl - 1);
            nbk = min(nbk, 4u * (uint32_t)nl);
        }
        *reinterpret_cast<uint4 *>(&L.bc[4 * lane]) = make_uint4(bc[0], bc[1], bc[2], bc[3]);
        if constexpr (MODE == COO_GROUP) group_rows(first, cb, nbk, k, L, lane);
        if constexpr (TILE)
            *reinterpret_cast<uint2 *>(&L.to[4 * lane]) = make_uint2(to[0] | (to[1] << 16), to[2] | (to[3] << 16));
        ends32[lane] = 0u;
        wave_sync();
        uint32_t p = incl - zs;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p += z[i];
            if (z[i] && mine) atomicOr(&ends32[(p - 1u) >> 5], 1u << ((p - 1u) & 31u));
        }
        wave_sync();
        // few windows in flight keep the tiles' common sweep of a large x
        // together (Balance::tile_windows)
        if (TILE && windows == 1)
            seg_windows<VT, IT, COMP, SEG_STRIPS, 1>(val + e, idx + e, T, nbk, 0u, k, x, acc, L, lane);
        else if (TILE && windows == 2)
            seg_windows<VT, IT, COMP, SEG_STRIPS, 2>(val + e, idx + e, T, nbk, 0u, k, x, acc, L, lane);
        else
            seg_windows<VT, IT, COMP, MODE == COO_STRIP ? SEG_COO : SEG_STRIPS, 4>(val + e, idx + e, T, nbk, 0u, k, x,
                                                                                   acc, L, lane);
        wave_sync();
        e += T;
        cb += nbk;
    }
}

// Bitmap or dense group of a strip, s >= 16.  Each lane owns cw consecutive
// row-major positions of the block (P = s / cw lanes per row); it accumulates its
// products in registers, the P lanes of a row are summed with DPP, and the
// first lane of the row adds the sum to the strip accumulator.
template <typename VT, typename BT, bool COMP>
__device__ __forceinline__ void bmdn_r1(MatPtr A_, int sc, uint32_t b0, uint32_t b1, uint64_t vb,
                               const double *__restrict__ x, const Acc &acc, int lane_)
{
    if (b0 >= b1) return;
    const MatPtr A = opaque_s(A_);
    const int lane = opaque_v(lane_);
    const int s = A->s, k = A->k;
    const uint32_t ss = (uint32_t)s * (uint32_t)s;
    const uint32_t cw = s >= 64 ? (uint32_t)s : ss / 64u;
    const int npass = (int)(ss / (64u * cw));
    const int P = (int)((uint32_t)s / cw);
    const int64_t n = A->n;
    const VT *__restrict__ val = glob<VT>(A->val[sc]);
#pragma unroll 1
    for (uint32_t b = b0; b < b1; b++) {
        const int64_t c0 = (int64_t)glob<BT>(A->bcol[sc])[b] * s;
        const uint64_t *__restrict__ words = glob<uint64_t>(A->bm_words) + (uint64_t)b * A->W;
        const uint64_t db = (uint64_t)b * ss;
#pragma unroll 1
        for (int q = 0; q < npass; q++) {
            const uint32_t pbase = ((uint32_t)q * 64u + (uint32_t)lane) * cw;
            const uint32_t row = pbase >> k, col0 = pbase & ((uint32_t)s - 1);
            const int64_t gc0 = c0 + col0;
            double hi = 0.0, lo = 0.0;
            if (sc == DENSE) {
                const VT *vp = val + db + pbase;
                // double2 loads of x need a 16-byte aligned x (a caller may pass
                // x + 1 of an array): otherwise the scalar walk below
                if (gc0 + (int64_t)cw <= n && (cw & 1) == 0 && x_aligned16(x)) {
#pragma unroll 4
                    for (uint32_t c = 0; c < cw; c += 2) {
                        const double2 xv = *reinterpret_cast<const double2 *>(x + gc0 + c);
                        double v0, v1;
                        if constexpr (sizeof(VT) == 8) {
                            const double2 vv = *reinterpret_cast<const double2 *>(vp + c);
                            v0 = vv.x;
                            v1 = vv.y;
                        } else {
                            const float2 vv = *reinterpret_cast<const float2 *>(vp + c);
                            v0 = vv.x;
                            v1 = vv.y;
                        }
                        acc_add<COMP>(hi, lo, v0, xv.x);
                        acc_add<COMP>(hi, lo, v1, xv.y);
                    }
                } else {
                    for (uint32_t c = 0; c < cw; c++)
                        if (gc0 + c < n) acc_add<COMP>(hi, lo, (double)vp[c], x[gc0 + c]);
                }
            } else {
                // bitmap: popcount of my positions -> value offset by a wave scan
                const uint32_t nw = cw > 64 ? cw / 64 : 1;
                const uint32_t w0 = pbase >> 6, sh = pbase & 63;
                const uint64_t m = cw >= 64 ? ~0ull : ((1ull << cw) - 1ull);
                uint32_t cnt = 0;
                for (uint32_t w = 0; w < nw; w++) cnt += __popcll((words[w0 + w] >> sh) & m);
                const uint32_t incl = wave_incl_scan_dpp(cnt);
                const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
                uint64_t off = vb + incl - cnt;
                for (uint32_t w = 0; w < nw; w++) {
                    uint64_t bits = (words[w0 + w] >> sh) & m;
                    const int64_t xb = gc0 + (int64_t)w * 64;
                    // four set bits per step so their loads are in flight together
                    while (bits) {
                        const uint32_t c0 = (uint32_t)__builtin_ctzll(bits);
                        bits &= bits - 1;
                        const bool h1 = bits != 0;
                        const uint32_t c1 = h1 ? (uint32_t)__builtin_ctzll(bits) : c0;
                        bits &= bits - 1;
                        const bool h2 = bits != 0;
                        const uint32_t c2 = h2 ? (uint32_t)__builtin_ctzll(bits) : c0;
                        bits &= bits - 1;
                        const bool h3 = bits != 0;
                        const uint32_t c3 = h3 ? (uint32_t)__builtin_ctzll(bits) : c0;
                        bits &= bits - 1;
                        const double v0 = (double)val[off];
                        const double v1 = (double)val[h1 ? off + 1 : off];
                        const double v2 = (double)val[h2 ? off + 2 : off];
                        const double v3 = (double)val[h3 ? off + 3 : off];
                        const double x0 = x[xb + c0], x1 = x[xb + c1], x2 = x[xb + c2], x3 = x[xb + c3];
                        acc_add<COMP>(hi, lo, v0, x0);
                        if (h1) acc_add<COMP>(hi, lo, v1, x1);
                        if (h2) acc_add<COMP>(hi, lo, v2, x2);
                        if (h3) acc_add<COMP>(hi, lo, v3, x3);
                        off += 1u + h1 + h2 + h3;
                    }
                }
                vb += tot;
            }
            group_reduce<COMP>(P, hi, lo);
            if ((lane & (P - 1)) == 0) {
                if constexpr (COMP) {
                    double s2, e2;
                    two_sum(acc.hi[row], hi, s2, e2);
                    acc.hi[row] = s2;
                    acc.lo[row] += lo + e2;
                } else {
                    acc.hi[row] += hi;
                }
            }
        }
    }
}

// Bitmap blocks of s <= 16 rows, or dense blocks of s <= 8: a lane takes one
// position, so a wave step covers 64 consecutive positions (a quarter of a
// 16-row block, one 8-row block, several smaller ones), four steps in flight.
// A bitmap lane's value follows from the set bits in the lanes before it; the
// s lanes of a row are summed with DPP and its first lane adds the sum to the
// strip accumulator.  Block columns and, in a group of T > 1 strips from I0 on,
// the strips' rows come from LDS, 256 blocks at a time.
// Bound: memory latency.  One block per step, as before, was two round trips
// per block: 2048^2 Laplacian s = 8 (a bitmap block per strip) 786 -> 114 us
// with groups of strips, banded n = 10^6 bandwidth 10 s = 8 220 -> 58 us.
template <typename VT, typename BT, bool COMP, int SC>
__device__ __forceinline__ void small_r1(MatPtr A_, uint32_t b0, uint32_t b1, uint32_t e, const double *__restrict__ x,
                                         const Acc &acc, WaveLds &L, int lane_, int64_t I0, int T_)
{
    if (b0 >= b1) return;
    constexpr int U = 4;
    const MatPtr A = opaque_s(A_);
    const int lane = opaque_v(lane_);
    const int k = A->k;
    const uint32_t smask = (1u << k) - 1u, pmask = (1u << (2 * k)) - 1u;
    const VT *__restrict__ val = glob<VT>(A->val[SC]);
    const BT *__restrict__ bcol = glob<BT>(A->bcol[SC]);
    const uint64_t *__restrict__ words = glob<uint64_t>(A->bm_words);
    const int64_t n = A->n;
    uint32_t first = ~0u;
    if (T_ > 1) first = group_first<SC>(A, I0, T_, lane);
#pragma unroll 1
    for (uint32_t cb = b0; cb < b1; cb += (uint32_t)kSegs) {
        const uint32_t nbk = min<uint32_t>(kSegs, b1 - cb);
        uint32_t bc[4];
        load4(bcol, cb, nbk, lane, bc);
        *reinterpret_cast<uint4 *>(&L.bc[4 * lane]) = make_uint4(bc[0] << k, bc[1] << k, bc[2] << k, bc[3] << k);
        if (T_ > 1) group_rows(first, cb, nbk, k, L, lane);
        else *reinterpret_cast<uint2 *>(&L.to[4 * lane]) = make_uint2(0u, 0u);
        wave_sync();
        const uint32_t P = nbk << (2 * k);  // positions of the chunk
#pragma unroll 1
        for (uint32_t q = 0; q < P; q += (uint32_t)(U * kWave)) {
            uint32_t bl[U], pos[U];
            bool on[U];
            double v[U], xv[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t pp = q + (uint32_t)(u * kWave + lane);
                on[u] = pp < P;
                bl[u] = min(pp, P - 1u) >> (2 * k);
                pos[u] = pp & pmask;
                if constexpr (SC == BITMAP) {
                    const uint64_t w = words[((uint64_t)(cb + bl[u]) * (uint64_t)((pmask >> 6) + 1u)) + (pos[u] >> 6)];
                    on[u] = on[u] && ((w >> (pos[u] & 63u)) & 1ull);
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t c = L.bc[bl[u]] + (pos[u] & smask);
                uint64_t off;
                if constexpr (SC == BITMAP) {
                    const uint64_t m = __ballot(on[u]);
                    off = e + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                    e += (uint32_t)__popcll(m);
                } else {
                    on[u] = on[u] && (int64_t)c < n;  // columns past n hold stored zeros; x is not read there
                    off = ((uint64_t)(cb + bl[u]) << (2 * k)) + pos[u];
                }
                v[u] = on[u] ? (double)val[off] : 0.0;
                xv[u] = on[u] ? x[c] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                double hi, lo;
                hi = prod<COMP>(v[u], xv[u], lo);
                row_reduce<COMP>(k, hi, lo);
                if ((pos[u] & smask) == 0 && q + (uint32_t)(u * kWave + lane) < P)
                    acc_atomic<COMP>(acc, (pos[u] >> k) + L.to[bl[u]], hi, lo);
            }
        }
        wave_sync();
    }
}

// Dense group of an S-row strip (S = 16 or 32), FP64 values, coalesced: wave
// step q reads positions q*128 + 2l, +1 of the block (1 KB contiguous); lane
// l always has columns 2(l % L), +1 (L = S/2 lanes per row) and rows
// q*(128/S) + l/L, so its x pair is read once per block and it keeps one
// accumulator per step over all the group's blocks; the L lanes of a row are
// summed with DPP at the end.  (Lanes owning S*S/64 consecutive positions
// made a load touch up to 64 lines: S = 32 streamed 3.8 TB/s, now 5.6.)
template <typename BT, int S>
__device__ __forceinline__ void dense_coal_r1(MatPtr A_, uint32_t b0, uint32_t b1, const double *__restrict__ x,
                                     const Acc &acc, int lane_)
{
    static_assert(S == 16 || S == 32, "S x S blocks of whole 128-position steps");
    constexpr int L = S / 2, NQ = S * S / 128, RQ = 128 / S;
    if (b0 >= b1) return;
    const MatPtr A = opaque_s(A_);
    const int lane = opaque_v(lane_);
    const double *__restrict__ val = glob<double>(A->val[DENSE]);
    const int64_t n = A->n;
    const int cl = 2 * (lane % L);
    const bool xal = x_aligned16(x);  // wave-uniform: x pairs as double2 loads or two scalar loads
    double a[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) a[q] = 0.0;
#pragma unroll 1
    for (uint32_t b = b0; b < b1; b++) {
        const int64_t c0 = (int64_t)glob<BT>(A->bcol[DENSE])[b] * S + cl;
        double x0 = 0.0, x1 = 0.0;  // columns past n hold stored zeros; x is not read there
        if (c0 + 1 < n && !xal) {
            x0 = x[c0];
            x1 = x[c0 + 1];
        } else if (c0 + 1 < n) {
            const double2 xv = *reinterpret_cast<const double2 *>(x + c0);
            x0 = xv.x;
            x1 = xv.y;
        } else if (c0 < n) {
            x0 = x[c0];
        }
        const double2 *__restrict__ vp = reinterpret_cast<const double2 *>(val + (uint64_t)b * (S * S)) + lane;
#pragma unroll
        for (int h = 0; h < NQ; h += 4) {  // at most four loads in flight (register budget)
            constexpr int H = NQ < 4 ? NQ : 4;
            double2 v[H];
#pragma unroll
            for (int q = 0; q < H; q++) v[q] = vp[(h + q) * 64];
#pragma unroll
            for (int q = 0; q < H; q++) a[h + q] = __builtin_fma(v[q].y, x1, __builtin_fma(v[q].x, x0, a[h + q]));
            __builtin_amdgcn_sched_barrier(0);  // keep the next loads behind these
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const double r = group_sum_dpp<L>(a[q]);
        if (lane % L == 0) acc.hi[q * RQ + lane / L] += r;
    }
}

// Dense group of a strip: the coalesced path for FP64 16- and 32-row blocks,
// position by position for smaller ones, the bitmap/dense walk otherwise.  The
// index types tell the block-size class at compile time (u8 indices: s <= 16,
// with u16 row pointers s = 16; u16 indices: s >= 32), so each kernel carries
// only the paths it can take.
template <typename VT, typename BT, typename IT, typename RT, bool COMP>
__device__ __forceinline__ void dense_r1(MatPtr A, uint32_t b0, uint32_t b1, const double *__restrict__ x,
                                         const Acc &acc, WaveLds &L, int lane)
{
    if constexpr (sizeof(RT) == 1) {
        small_r1<VT, BT, COMP, DENSE>(A, b0, b1, 0u, x, acc, L, lane, 0, 1);
        return;
    }
    if constexpr (sizeof(VT) == 8 && !COMP && sizeof(IT) == 2) {
        if (A->s == 32) {
            dense_coal_r1<BT, 32>(A, b0, b1, x, acc, lane);
            return;
        }
    }
    if constexpr (sizeof(VT) == 8 && !COMP && sizeof(IT) == 1) {
        dense_coal_r1<BT, 16>(A, b0, b1, x, acc, lane);
        return;
    }
    bmdn_r1<VT, BT, COMP>(A, DENSE, b0, b1, 0, x, acc, lane);
}

// Bitmap group of a strip: position by position up to s = 8; a 16-row block's
// lanes own four positions each in the lane walk and have their loads in one
// round trip as well (27-point stencil 100^3 s = 16, FP32 values: 289 us, and
// 508 us position by position).
template <typename VT, typename BT, typename RT, bool COMP>
__device__ __forceinline__ void bitmap_r1(MatPtr A, uint32_t b0, uint32_t b1, uint32_t e, const double *__restrict__ x,
                                          const Acc &acc, WaveLds &L, int lane)
{
    if constexpr (sizeof(RT) == 1) small_r1<VT, BT, COMP, BITMAP>(A, b0, b1, e, x, acc, L, lane, 0, 1);
    else bmdn_r1<VT, BT, COMP>(A, BITMAP, b0, b1, e, x, acc, lane);
}

// Workgroups are dispatched to the 8 XCDs round-robin.  Renumber them so that
// each XCD (and its L2) receives runs of kRun consecutive work items (the x
// windows of neighbouring strips stay in one L2) while the runs rotate over
// the XCDs (a skewed range, e.g. the units of heavy strips, is still spread
// over all of them).  A tail shorter than 8 runs keeps the dispatch order.
__device__ inline int64_t xcd_block_id()
{
    constexpr int64_t kXcd = 8, kRun = 32;
    const int64_t nb = gridDim.x, b = blockIdx.x;
    const int64_t full = (nb / (kXcd * kRun)) * (kXcd * kRun);
    if (b >= full) return b;
    const int64_t x = b % kXcd, i = b / kXcd;
    return ((i / kRun) * kXcd + x) * kRun + (i % kRun);
}

// One work item of one matrix (see Balance): the wave accumulates in acc_buf
// (s doubles, 2s when compensated) and writes y rows or a unit's partials.
// Work items: items [0, n_light) are light items -- whole strips light[p] for
// p in [pack[item], pack[item + 1]) (p = item without pack; strip p without
// light) -- whose rows are written to y; items n_light + u are
// units u of heavy strips: one scheme group's block range, whose partial sums
// go to part[u] and are combined by k_spmv_fixup.
// TL: 0 the matrix is not tiled, 1 it is, 2 either (read from B.tiled); the
// single-matrix kernels are compiled for 0 or 1 so that each carries only one
// of the light-item paths (scalar-register pressure).
template <typename VT, typename BT, typename IT, typename RT, bool COMP, int TL = 2>
__device__ __forceinline__ void spmv_item(MatPtr A, BalPtr B, int64_t item, const double *__restrict__ x,
                                 double *__restrict__ y, double alpha, double beta, double *acc_buf, WaveLds &L,
                                 int lane)
{
    const int s = A->s;
    Acc acc;
    acc.hi = acc_buf;
    acc.lo = COMP ? acc_buf + 256 : nullptr;
    auto clear = [&](int rows) {
        for (int i = lane; i < rows; i += kWave) {
            acc.hi[i] = 0.0;
            if constexpr (COMP) acc.lo[i] = 0.0;
        }
        wave_sync();
    };
    if (item < B->n_light) {
        // light item: light strips at positions [p0, p1) of the light list
        uint32_t p0 = (uint32_t)item, p1 = (uint32_t)item + 1u;
        if (B->pack) {
            p0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)glob<uint32_t>(B->pack)[item]);
            p1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)glob<uint32_t>(B->pack)[item + 1]);
        }
        const bool tiled = TL == 1 || (TL == 2 && B->tiled);
        const int T = (int)(p1 - p0);
        const uint32_t *light = glob<uint32_t>(B->light);
        const int64_t I = light ? (int64_t)__builtin_amdgcn_readfirstlane((int)light[p0]) : (int64_t)p0;
        uint32_t tb0, tb1, te0, csr = 1;  // the item's COO blocks; T > 1: it has CSR blocks
        if (tiled) {
            const uint32_t *R = glob<uint32_t>(B->coo_rng) + (uint64_t)item * 4;
            tb0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)R[0]);
            tb1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)R[1]);
            te0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)R[2]);
            csr = (uint32_t)__builtin_amdgcn_readfirstlane((int)R[3]);
        } else {
            tb0 = glob<uint32_t>(A->sptr[COO])[I];
            tb1 = glob<uint32_t>(A->sptr[COO])[I + T];
            te0 = glob<uint32_t>(A->eptr[COO])[I];
        }
        // all bounds first: one round trip (a group's strips are consecutive;
        // a tile without CSR blocks does not use these)
        const int64_t Ie = csr ? I + T : I;
        const uint32_t r0 = glob<uint32_t>(A->sptr[CSR])[I], r1 = glob<uint32_t>(A->sptr[CSR])[Ie];
        const uint32_t re = glob<uint32_t>(A->eptr[CSR])[I];
        if (T > 1) {
            // several strips: a tile (COO blocks only), or a group of
            // consecutive strips; rows (position << k) + lrow
            const int rows = T * s;
            clear(rows);
            if (tiled) coo_r1<VT, BT, IT, COMP, COO_TILE>(A, tb0, tb1, te0, x, acc, L, lane, B->tile_windows);
            else coo_r1<VT, BT, IT, COMP, COO_GROUP>(A, tb0, tb1, te0, x, acc, L, lane, 4, I, T);
            csr_r1<VT, BT, RT, COMP>(A, r0, r1, re, x, acc, L, lane, I, T);
            if constexpr (sizeof(IT) == 1) {  // s <= 16
                wave_sync();
                small_r1<VT, BT, COMP, BITMAP>(A, glob<uint32_t>(A->sptr[BITMAP])[I], glob<uint32_t>(A->sptr[BITMAP])[Ie],
                                               glob<uint32_t>(A->eptr[BITMAP])[I], x, acc, L, lane, I, T);
            }
            if constexpr (sizeof(RT) == 1) {  // s <= 8
                wave_sync();
                small_r1<VT, BT, COMP, DENSE>(A, glob<uint32_t>(A->sptr[DENSE])[I], glob<uint32_t>(A->sptr[DENSE])[Ie], 0u,
                                              x, acc, L, lane, I, T);
            }
            wave_sync();
            for (int r = lane; r < rows; r += kWave) {
                const int64_t gr = (csr ? I + (r >> A->k) : (int64_t)light[p0 + (uint32_t)(r >> A->k)]) * s +
                                   (r & (s - 1));
                if (gr < A->m) {
                    double a = acc.hi[r];
                    if constexpr (COMP) a += acc.lo[r];
                    y[gr] = (beta == 0.0) ? alpha * a : alpha * a + beta * y[gr];
                }
            }
            wave_sync();
            return;
        }
        const uint32_t m0 = glob<uint32_t>(A->sptr[BITMAP])[I], m1 = glob<uint32_t>(A->sptr[BITMAP])[I + 1];
        const uint32_t me = glob<uint32_t>(A->eptr[BITMAP])[I];
        const uint32_t d0 = glob<uint32_t>(A->sptr[DENSE])[I], d1 = glob<uint32_t>(A->sptr[DENSE])[I + 1];
        clear(s);
        coo_r1<VT, BT, IT, COMP>(A, tb0, tb1, te0, x, acc, L, lane);
        csr_r1<VT, BT, RT, COMP>(A, r0, r1, re, x, acc, L, lane);
        wave_sync();
        bitmap_r1<VT, BT, RT, COMP>(A, m0, m1, me, x, acc, L, lane);
        dense_r1<VT, BT, IT, RT, COMP>(A, d0, d1, x, acc, L, lane);
        wave_sync();
        for (int r = lane; r < s; r += kWave) {
            const int64_t gr = I * s + r;
            if (gr >= A->m) break;
            double a = acc.hi[r];
            if constexpr (COMP) a += acc.lo[r];
            y[gr] = (beta == 0.0) ? alpha * a : alpha * a + beta * y[gr];
        }
        wave_sync();
    } else {
        const int64_t u = item - B->n_light;
        const uint32_t *U = glob<uint32_t>(B->units) + u * 4;
        const uint32_t sc = U[0] & 3u, b0 = U[1], b1 = U[2], e0 = U[3];
        clear(s);
        // constant scheme arguments: the descriptor's per-scheme arrays are
        // then indexed statically (a runtime index would force a local copy
        // of the descriptor, as in the batched kernel, into scratch memory)
        if (sc == COO)
            coo_r1<VT, BT, IT, COMP>(A, b0, b1, e0, x, acc, L, lane);
        else if (sc == CSR)
            csr_r1<VT, BT, RT, COMP>(A, b0, b1, e0, x, acc, L, lane);
        else if (sc == BITMAP)
            bitmap_r1<VT, BT, RT, COMP>(A, b0, b1, e0, x, acc, L, lane);
        else
            dense_r1<VT, BT, IT, RT, COMP>(A, b0, b1, x, acc, L, lane);
        wave_sync();
        double *part = glob_rw(B->part) + u * (size_t)s * (COMP ? 2 : 1);
        for (int r = lane; r < s; r += kWave) {
            part[r] = acc.hi[r];
            if constexpr (COMP) part[s + r] = acc.lo[r];
        }
    }
    wave_sync();  // the next item reuses the LDS buffers
}

struct StripArgs {
    DevMat A;
    Balance B;
    const double *x;
    double *y;
    double alpha, beta;
};

// Waves per SIMD at least (registers): FP32 values at s <= 16 wait on memory
// and took 81 registers, five waves (27-point stencil 160^3 s = 16 tiled 1440
// us, six 1257; banded n = 10^6 bandwidth 10 s = 8 107 -> 90; R-MAT scale 20
// s = 16 tiled pays 115 -> 121).  At s >= 32 a sixth wave costs more than it
// gives (2e6 uniform random columns, 24 a row, s = 64 tiled 413 -> 464).
template <typename IT, bool COMP>
constexpr int strip_min_waves() { return COMP && sizeof(IT) == 1 ? 6 : 1; }

template <typename VT, typename BT, typename IT, typename RT, bool COMP, bool TILED>
__global__ __launch_bounds__(64 * kStripWaves, (strip_min_waves<IT, COMP>())) void k_spmv_strip(StripArgs)
{
    constexpr int kWaves = kStripWaves;
    // s rows, or a tile's (kTileRows; kTileRowsComp compensated, lo half at +256)
    static_assert(kTileRowsComp == 256 && kGroupRows == 256 && kTileRows >= 512, "accumulator layout");
    __shared__ double s_acc[kWaves][TILED || COMP ? kTileRows : kGroupRows];
    __shared__ __align__(16) WaveLds s_lds[kWaves];
    // the arguments, where the launch put them (the struct is the only one)
    const auto *P = (const __attribute__((address_space(4))) StripArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    const BalPtr B = &P->B;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    int64_t item = xcd_block_id() * kWaves + wave;
    if (B->order) {  // a slot table (column panels: items per XCD; tiles: launch order)
        const uint32_t o = glob<uint32_t>(B->order)[(int64_t)blockIdx.x * kWaves + wave];
        if (o == kNoItem) return;
        item = (int64_t)__builtin_amdgcn_readfirstlane((int)o);
    }
    if (item >= B->n_light + B->n_units) return;  // whole wave leaves; no workgroup barriers below
    spmv_item<VT, BT, IT, RT, COMP, TILED ? 1 : 0>(&P->A, B, item, glob<double>(P->x), glob_rw(P->y), P->alpha,
                                                   P->beta, s_acc[wave], s_lds[wave], lane);
}

// ===========================================================================
// Symmetric storage (one triangle T stored): the main pass computes
// y = alpha*T*x + beta*y, this pass adds scale * T_off^T * x (scale = alpha,
// or -alpha for skew-symmetric; T_off = T without its diagonal): for every
// stored entry (i, j), i != j, y[j] += scale * a_ij * x[i], by global FP64
// atomics (entries of a strip scatter over the column range).  FP64 values.
// ===========================================================================

// A wave takes one strip (or unit).  Its x rows are kept in LDS, and the
// products (scale v) x (scale x may leave the range where scale v does not) of
// up to kTransAcc / s blocks are summed by column in LDS before they are added
// to y, 64 consecutive columns per wave instruction.  Scattered COO blocks are
// added entry by entry, 256 blocks at a time (trans_coo).
// Bound: the global adds, which the fabric takes one request at a time.  With
// an add for every entry (about 31 requests per wave instruction) the 27-point
// stencil 99^3, s = 64, one triangle took 262 us for this pass, now about 70.
constexpr int kTransAcc = 512;

struct TransArgs {
    DevMat A;
    Balance B;
    const double *x;
    double *y;
    int64_t ldx, ldy;
    double scale;
};

struct TransLds {
    double acc[kTransAcc];  // sums by column, s per block of the chunk
    double xs[256];         // x of the strip's rows
    WaveLds w;
};

// Sums of nb blocks from cb on to y, cleared.
template <typename BT>
__device__ __forceinline__ void trans_flush(const BT *__restrict__ bcol, uint32_t cb, uint32_t nb, int k, double *y,
                                            int64_t ldy, TransLds &L, int lane)
{
    wave_sync();
#pragma unroll 1
    for (uint32_t i = (uint32_t)lane; i < nb << k; i += kWave) {
        const double v = L.acc[i];
        if (v != 0.0) {
            L.acc[i] = 0.0;
            const int64_t gc = ((int64_t)bcol[cb + (i >> k)] << k) + (i & ((1u << k) - 1u));
            atomicAdd(&y[gc * ldy], v);
        }
    }
    wave_sync();
}

// Entries [vp, vp + T) of a chunk (COO or CSR: see seg_windows).  L.w.bc holds
// a segment's first column (direct) or its block's first sum; L.w.to the
// block's diagonal flag, for CSR the row with the flag in bit 15.
template <typename IT, bool CSRM>
__device__ __forceinline__ void trans_windows(const double *__restrict__ vp, const IT *__restrict__ ip, uint32_t T,
                                              uint32_t nseg, uint32_t before, int k, double *y, int64_t ldy,
                                              double scale, bool direct, TransLds &L, int lane)
{
    constexpr int U = 4;
    const uint32_t smask = (1u << k) - 1u;
#pragma unroll 1
    for (uint32_t q = 0; q < T; q += (uint32_t)(U * kWave)) {
        uint32_t id[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t t = min(q + (uint32_t)(u * kWave + lane), T - 1u);
            id[u] = ip[t];
            v[u] = vp[t];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (q + (uint32_t)(u * kWave) >= T) break;  // uniform
            const uint64_t m = L.w.ends[q / kWave + (uint32_t)u];
            const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
            const uint32_t own = min(__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, before)), nseg - 1u);
            before += (uint32_t)__popc(lo) + (uint32_t)__popc(hi);
            const uint32_t to = L.w.to[own];
            const uint32_t r = CSRM ? to & 0x7FFFu : id[u] >> k, c = CSRM ? id[u] : id[u] & smask;
            const bool diag = (CSRM ? to >> 15 : to) && r == c;
            if (q + (uint32_t)(u * kWave + lane) < T && !diag) {
                const double p = (scale * v[u]) * L.xs[r];
                if (direct) atomicAdd(&y[(int64_t)(L.w.bc[own] + c) * ldy], p);
                else atomicAdd(&L.acc[L.w.bc[own] + c], p);
            }
        }
    }
}

// COO blocks.  The sums by column pay where the chunk of kTransAcc / s blocks
// holds entries for half of its columns or more; below, the chunk is a handful
// of entries between two passes over the sums, and the entries are added to y
// as they come, in chunks of up to 256 blocks that end at the next block that
// holds entries for half of its columns.  With the sums everywhere (a mean of two entries a block over
// the matrix) one triangle of 2e5 uniform random columns, 8 a row, took 1255
// us at s = 256 (55 now), 32 a row at s = 128 1770 us (174), R-MAT scale 16 at
// s = 256 370 us (76).  The line at s / 4: uniform n = 2e4, 32 a row, s = 256
// 135 us (50 here); at 3 s / 4: stencil 99^3 s = 256 96 us (74 here).  Up to
// s = 8 a block's columns lie in one line, and the line is at 3 s / 4: R-MAT
// scale 16 s = 8 240 us at s / 2, 235 here; never: an arrow of n = 1e5, whose
// strips all add to column 0, 1211 us, 161 here.
template <typename BT, typename IT>
__device__ __forceinline__ void trans_coo(MatPtr A_, uint32_t b0, uint32_t b1, uint32_t e, int64_t I, double *y,
                                          int64_t ldy, double scale, TransLds &L, int lane)
{
    if (b0 >= b1) return;
    const MatPtr A = opaque_s(A_);
    const int k = A->k;
    const double *__restrict__ val = glob<double>(A->val[COO]);
    const IT *__restrict__ idx = glob<IT>(A->coo_idx);
    const uint16_t *__restrict__ z1 = glob<uint16_t>(A->z1[COO]);
    const BT *__restrict__ bcol = glob<BT>(A->bcol[COO]);
    uint32_t *ends32 = reinterpret_cast<uint32_t *>(L.w.ends);
    const uint32_t cap = min((uint32_t)kTransAcc >> k, (uint32_t)kSegs);
    const uint32_t full = k > 3 ? 1u << (k - 1) : max(2u, (3u << k) >> 2);
    uint32_t cb = b0, look = (uint32_t)kSegs;  // blocks to look at
#pragma unroll 1
    while (cb < b1) {
        uint32_t nbk = min(look, b1 - cb), z[4], bc[4], zs = 0;
        load4(z1, cb, nbk, lane, z);
        load4(bcol, cb, nbk, lane, bc);
        // the first `cap` blocks' entries, and the first such block after them
        uint32_t f = 4;
#pragma unroll
        for (int i = 3; i >= 0; i--) {
            const uint32_t j = 4u * (uint32_t)lane + (uint32_t)i;
            z[i] = j < nbk ? z[i] + 1u : 0u;
            zs += z[i];
            if (j >= cap && z[i] >= full) f = (uint32_t)i;
        }
        uint32_t incl = wave_incl_scan_dpp(zs);
        const uint32_t first = cap < 4u ? (uint32_t)__builtin_amdgcn_readfirstlane((int)(z[0] + z[1]))
                                        : (uint32_t)__builtin_amdgcn_readlane((int)incl, (int)(cap / 4u) - 1);
        const uint32_t ncap = min(cap, nbk);
        const bool direct = first < ncap * full;  // uniform; (so a chunk always holds a block)
        if (direct) {
            const uint64_t any = __ballot(f < 4u);
            if (any) {
                const int l = __builtin_ctzll(any);
                nbk = 4u * (uint32_t)l + (uint32_t)__builtin_amdgcn_readlane((int)f, l);
            }
        } else {
            nbk = ncap;
        }
        look = direct ? (uint32_t)kSegs : cap;
        // without the blocks from nbk on (the sums of later lanes are not used)
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (4u * (uint32_t)lane + (uint32_t)i >= nbk) {
                incl -= z[i];
                zs -= z[i];
                z[i] = 0u;
            }
        uint32_t T = (uint32_t)__builtin_amdgcn_readlane((int)incl, (int)((nbk - 1u) >> 2));
        bool mine = true;
        if (T > (uint32_t)kMaskEnts) {  // uniform: take the lanes whose blocks fit
            mine = incl <= (uint32_t)kMaskEnts;
            const int nl = __popcll(__ballot(mine));
            T = (uint32_t)__builtin_amdgcn_readlane((int)incl, nl - 1);
            nbk = min(nbk, 4u * (uint32_t)nl);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t j = 4u * (uint32_t)lane + (uint32_t)i;
            L.w.bc[j] = direct ? bc[i] << k : j << k;
            L.w.to[j] = (int64_t)bc[i] == I;
        }
        ends32[lane] = 0u;
        wave_sync();
        uint32_t p = incl - zs;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p += z[i];
            if (z[i] && mine) atomicOr(&ends32[(p - 1u) >> 5], 1u << ((p - 1u) & 31u));
        }
        wave_sync();
        trans_windows<IT, false>(val + e, idx + e, T, nbk, 0u, k, y, ldy, scale, direct, L, lane);
        if (!direct) trans_flush(bcol, cb, nbk, k, y, ldy, L, lane);
        wave_sync();
        e += T;
        cb += nbk;
    }
}

template <typename BT, typename RT>
__device__ __forceinline__ void trans_csr(MatPtr A_, uint32_t b0, uint32_t b1, uint32_t e, int64_t I, double *y,
                                          int64_t ldy, double scale, TransLds &L, int lane)
{
    if (b0 >= b1) return;
    const MatPtr A = opaque_s(A_);
    const int k = A->k;
    const double *__restrict__ val = glob<double>(A->val[CSR]);
    const uint8_t *__restrict__ ccol = glob<uint8_t>(A->csr_col);
    const RT *__restrict__ rowptr = glob<RT>(A->csr_rowptr);
    const BT *__restrict__ bcol = glob<BT>(A->bcol[CSR]);
    uint32_t *ends32 = reinterpret_cast<uint32_t *>(L.w.ends);
    const uint32_t nb = (uint32_t)kSegs >> k;  // blocks per chunk (256 rows, as csr_r1)
    const uint32_t j = (4u * (uint32_t)lane) >> k, r0 = (4u * (uint32_t)lane) & ((1u << k) - 1u);
#pragma unroll 1
    for (uint32_t cb = b0; cb < b1; cb += nb) {
        uint32_t a[5] = {0, 0, 0, 0, 0}, diag = 0;
        if (cb + j < b1) {
            const RT *__restrict__ rp = rowptr + ((uint64_t)(cb + j) * (uint64_t)((1u << k) + 1u) + r0);
#pragma unroll
            for (int i = 0; i < 5; i++) a[i] = (uint32_t)rp[i];
            diag = (int64_t)bcol[cb + j] == I ? 0x8000u : 0u;
        }
        uint32_t rows = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) rows += a[i + 1] != a[i];
        const uint32_t mine = (a[4] - a[0]) | (rows << 16);
        const uint32_t incl = wave_incl_scan_dpp(mine);
        const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        const uint32_t T = tot & 0xFFFFu, nseg = tot >> 16;
        const uint32_t p0 = ((incl - mine) & 0xFFFFu) - a[0];
        uint32_t o = (incl - mine) >> 16;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (a[i + 1] != a[i]) {
                L.w.bc[o] = j << k;
                L.w.to[o] = (uint16_t)(diag | (r0 + (uint32_t)i));
                o++;
            }
#pragma unroll 1
        for (uint32_t w = 0; w < T; w += (uint32_t)kMaskEnts) {
            const uint32_t Tw = min(T - w, (uint32_t)kMaskEnts);
            ends32[lane] = 0u;
            wave_sync();
            uint32_t before = 0;  // rows that end before entry w
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (a[i + 1] != a[i]) {
                    const uint32_t last = p0 + a[i + 1] - 1u;
                    before += last < w;
                    if (last - w < Tw) atomicOr(&ends32[(last - w) >> 5], 1u << ((last - w) & 31u));
                }
            if (w) before = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan_dpp(before), kWave - 1);
            wave_sync();
            trans_windows<uint8_t, true>(val + (e + w), ccol + (e + w), Tw, nseg, before, k, y, ldy, scale, false, L,
                                         lane);
            wave_sync();
        }
        trans_flush(bcol, cb, min(nb, b1 - cb), k, y, ldy, L, lane);
        e += T;
    }
}

// Bitmap or dense blocks, one at a time, lanes over the positions.
template <typename BT, int SC>
__device__ __forceinline__ void trans_bmdn(MatPtr A_, uint32_t b0, uint32_t b1, uint32_t e, int64_t I, double *y,
                                           int64_t ldy, double scale, TransLds &L, int lane)
{
    if (b0 >= b1) return;
    const MatPtr A = opaque_s(A_);
    const int k = A->k;
    const uint32_t ss = 1u << (2 * k), smask = (1u << k) - 1u, W = ss >= 64u ? ss >> 6 : 1u;
    const double *__restrict__ val = glob<double>(A->val[SC]);
    const uint64_t *__restrict__ words = glob<uint64_t>(A->bm_words);
    const BT *__restrict__ bcol = glob<BT>(A->bcol[SC]);
    const int64_t n = A->n;
#pragma unroll 1
    for (uint32_t b = b0; b < b1; b++) {
        const int64_t J = (int64_t)bcol[b];
#pragma unroll 1
        for (uint32_t w = 0; w < W; w++) {
            const uint32_t pos = w * 64u + (uint32_t)lane;
            const uint32_t r = pos >> k, c = pos & smask;
            bool on = pos < ss;
            uint64_t off = ((uint64_t)b << (2 * k)) + pos;
            if constexpr (SC == BITMAP) {
                const uint64_t word = words[(uint64_t)b * W + w];
                on = on && ((word >> lane) & 1ull);
                off = e + __popcll(word & lanemask_lt());
                e += (uint32_t)__popcll(word);
            } else {
                on = on && (J << k) + c < n;
            }
            const double v = on ? val[off] : 0.0;
            // zeros fill a dense block where it has no entry: not a product
            // (x there may be infinite)
            if (SC == DENSE) on = on && v != 0.0;
            if (on && !(J == I && r == c)) atomicAdd(&L.acc[c], (scale * v) * L.xs[r]);
        }
        trans_flush(bcol, b, 1u, k, y, ldy, L, lane);
    }
}

template <typename BT, typename IT, typename RT>
__global__ __launch_bounds__(64 * kStripWaves) void k_spmv_trans(TransArgs)
{
    __shared__ __align__(16) TransLds s_lds[kStripWaves];
    const auto *P = (const __attribute__((address_space(4))) TransArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    const MatPtr A = &P->A;
    const BalPtr B = &P->B;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * kStripWaves + wave;
    if (item >= B->n_lstrips + B->n_units) return;
    TransLds &L = s_lds[wave];
    const int s = A->s;
    const double *x = glob<double>(P->x);
    double *y = glob_rw(P->y);
    const int64_t ldy = P->ldy;
    const double scale = P->scale;
    int64_t I;
    uint32_t sc = 4, b0 = 0, b1 = 0, e0 = 0;  // scheme 4: a whole strip
    if (item < B->n_lstrips) {
        const uint32_t *light = glob<uint32_t>(B->light);
        I = light ? (int64_t)__builtin_amdgcn_readfirstlane((int)light[item]) : item;
    } else {
        const uint32_t *U = glob<uint32_t>(B->units) + (item - B->n_lstrips) * 4;
        const uint32_t u0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)U[0]);
        I = (int64_t)(u0 >> 2);
        sc = u0 & 3u;
        b0 = U[1];
        b1 = U[2];
        e0 = U[3];
    }
    for (int i = lane; i < kTransAcc; i += kWave) L.acc[i] = 0.0;
    for (int r = lane; r < s; r += kWave) {
        const int64_t gr = I * s + r;
        L.xs[r] = gr < A->m ? x[gr * P->ldx] : 0.0;
    }
    wave_sync();
    // (constant scheme arguments: see spmv_item)
    auto range = [&](int q, uint32_t &f, uint32_t &l, uint32_t &e) {
        f = sc == 4 ? glob<uint32_t>(A->sptr[q])[I] : b0;
        l = sc == 4 ? glob<uint32_t>(A->sptr[q])[I + 1] : b1;
        e = sc == 4 ? glob<uint32_t>(A->eptr[q])[I] : e0;
    };
    uint32_t f, l, e;
    if (sc == 4 || sc == COO) {
        range(COO, f, l, e);
        trans_coo<BT, IT>(A, f, l, e, I, y, ldy, scale, L, lane);
    }
    if (sc == 4 || sc == CSR) {
        range(CSR, f, l, e);
        trans_csr<BT, RT>(A, f, l, e, I, y, ldy, scale, L, lane);
    }
    if (sc == 4 || sc == BITMAP) {
        range(BITMAP, f, l, e);
        trans_bmdn<BT, BITMAP>(A, f, l, e, I, y, ldy, scale, L, lane);
    }
    if (sc == 4 || sc == DENSE) {
        range(DENSE, f, l, e);
        trans_bmdn<BT, DENSE>(A, f, l, e, I, y, ldy, scale, L, lane);
    }
}

// Many matrices in one launch: the waves take the global items [0, G), wave w
// items w, w + W, ... (W = all waves of the grid); item_mat[g] names the
// matrix of item g, whose index-type combination (batch_code) selects the
// decode (a uniform branch), so one launch serves every member.  FP64
// values.  TIMED: each wave also adds the shader-clock cycles of its item to
// cyc[matrix] (the per-matrix cost inside a full launch).
template <bool TIMED, bool COMP>
// (6 waves per SIMD asked of the register allocator: 86 VGPRs allowed 5; the
// 2000-matrix batch of tuned picks 6.11 -> 5.96 ms, plain s = 64 8.98 ->
// 9.00 ms)
__global__ __launch_bounds__(256, 6) void k_batch_spmv(const BatchEntry *__restrict__ E,
                                                    const uint32_t *__restrict__ item_mat, int64_t g0, int64_t G,
                                                    double alpha, double beta, unsigned long long *cyc)
{
    using VT = typename std::conditional<COMP, float, double>::type;
    constexpr int kWaves = 4;
    __shared__ double s_acc[kWaves][kTileRows];
    __shared__ __align__(16) WaveLds s_lds[kWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t nw = (int64_t)gridDim.x * kWaves;
#pragma unroll 1
    for (int64_t g = g0 + (int64_t)blockIdx.x * kWaves + wave; g < G; g += nw) {
        const int mat = __builtin_amdgcn_readfirstlane((int)item_mat[g]);
        // the table is read-only during the launch: constant address space
        const auto *e = (const __attribute__((address_space(4))) BatchEntry *)(E + mat);
        const double *x = glob<double>(e->x);
        double *y = glob_rw(e->y);
        long long t0 = 0;
        if constexpr (TIMED) t0 = clock64();
        const int64_t it = g - e->item0;
        double *sa = s_acc[wave];
        WaveLds &sl = s_lds[wave];
        switch (e->code) {  // batch_code: (bcol u32 ? 3 : 0) + (s <= 8 ? 0 : s <= 16 ? 1 : 2)
        case 0:
            spmv_item<VT, uint16_t, uint8_t, uint8_t, COMP>(&e->A, &e->B, it, x, y, alpha, beta, sa, sl, lane);
            break;
        case 1:
            spmv_item<VT, uint16_t, uint8_t, uint16_t, COMP>(&e->A, &e->B, it, x, y, alpha, beta, sa, sl, lane);
            break;
        case 2:
            spmv_item<VT, uint16_t, uint16_t, uint16_t, COMP>(&e->A, &e->B, it, x, y, alpha, beta, sa, sl, lane);
            break;
        case 3:
            spmv_item<VT, uint32_t, uint8_t, uint8_t, COMP>(&e->A, &e->B, it, x, y, alpha, beta, sa, sl, lane);
            break;
        case 4:
            spmv_item<VT, uint32_t, uint8_t, uint16_t, COMP>(&e->A, &e->B, it, x, y, alpha, beta, sa, sl, lane);
            break;
        default:
            spmv_item<VT, uint32_t, uint16_t, uint16_t, COMP>(&e->A, &e->B, it, x, y, alpha, beta, sa, sl, lane);
            break;
        }
        if constexpr (TIMED) {
            const long long t1 = clock64();
            if (lane == 0) atomicAdd(&cyc[mat], (unsigned long long)(t1 - t0));
        }
    }
}

// Rows [r0, r0 + rs) of one heavy strip I: y = alpha * (sum of the partial
// rows of units [u0, u0 + nu)) + beta * y, by a workgroup of kFixThreads
// threads.  The L = kFixThreads / rs threads of row r take units l, l + L, l + 2L, ... in
// kFixChains interleaved chains (that many loads in flight per thread); the
// chains and then the L threads are combined in a fixed order, so the sum
// does not depend on timing.  Partials of unit u: part[u * s * (COMP ? 2 : 1)
// + r] (+ s: the compensation terms).
// (R-MAT scale 22 at s = 256: the heaviest strip holds 584 units and sets the
// pass's length.  SpMV 0.545 ms with 512 threads x 4 chains, 0.532 ms with
// 256 x 16; 256 x 8 and 512 x 16 are in between, 32 chains spill: 0.61+ ms.
// 1024 threads x 4 chains was slower than 512 x 4.)  With compensated
// partials (two loads and a TwoSum per chain step) 16 chains do not stay in
// registers and the loads serialise: fix-up 285 us with 16 chains, 77 us with
// 8, 119 us with 4 (FP64 partials: 38 / 58 / 82 us).
#ifndef ABHSF_FIX_THREADS
#define ABHSF_FIX_THREADS 256
#endif
constexpr int kFixThreads = ABHSF_FIX_THREADS;
static_assert(kFixThreads >= 256, "at least one thread per row of a 256-row strip");
#ifndef ABHSF_FIX_CHAINS
#define ABHSF_FIX_CHAINS 16
#endif
template <bool COMP>
constexpr int kFixChains = COMP ? ABHSF_FIX_CHAINS / 2 : ABHSF_FIX_CHAINS;
static_assert(kFixChains<true> >= 4, "a quarter round of the fix-up takes one chain at least");
// Rows per fix-up workgroup: a strip of s > kFixRows rows is summed by s /
// kFixRows workgroups, kFixThreads / kFixRows threads per row.  R-MAT scale
// 22 at s = 256 (heaviest strip 585 units), fix-up with 256 / 128 / 64-row
// slices: FP64 39 / 31.5 / 36 us, compensated 91 / 48 / 40 us.
template <bool COMP>
constexpr int kFixRows = COMP ? 64 : 128;
static_assert(kFixThreads % 128 == 0, "whole threads per row");
// A heavy strip whose units would leave more than kFixUnits of them to each
// thread gets narrower slices (rows halved down to kFixRowsMin, threads per
// row doubled): the strips with the most units set the pass's length.
#ifndef ABHSF_FIX_UNITS
#define ABHSF_FIX_UNITS 32
#endif
constexpr int kFixUnits = ABHSF_FIX_UNITS;
constexpr int kFixRowsMin = 16;

template <bool COMP>
__device__ inline void fix_add(double &hi, double &lo, double v, double vlo)
{
    if constexpr (COMP) {
        double s2, e2;
        two_sum(hi, v, s2, e2);
        hi = s2;
        lo += vlo + e2;
    } else {
        hi += v;
    }
}

// One round of the fix-up's chains 0 .. W - 1 (units u + j * L; a chain past
// nu reads unit l and adds 0).
template <bool COMP, int W>
__device__ inline void fix_round(const double *__restrict__ part, size_t stride, uint32_t u0, uint32_t u, uint32_t l,
                                 uint32_t L, uint32_t nu, int s, int r, double *hi, double *lo)
{
#pragma unroll
    for (int j = 0; j < W; j++) {
        const uint32_t uj = u + (uint32_t)j * L;
        const bool ok = uj < nu;
        const double *p = part + (size_t)(u0 + (ok ? uj : l)) * stride;
        const double v = p[r], vlo = COMP ? p[s + r] : 0.0;
        fix_add<COMP>(hi[j], lo[j], ok ? v : 0.0, ok ? vlo : 0.0);
    }
}

template <bool COMP>
__device__ inline void fixup_strip(int s, int rs, int r0, int64_t m, int64_t I, const double *__restrict__ part,
                                   uint32_t u0, uint32_t nu, double *__restrict__ y, double alpha, double beta,
                                   double *sh)
{
    const uint32_t L = (uint32_t)(kFixThreads / rs);
    // consecutive threads take consecutive rows of one unit (coalesced loads)
    const int r = r0 + (int)(threadIdx.x % (uint32_t)rs);
    const uint32_t l = threadIdx.x / (uint32_t)rs;
    const size_t stride = (size_t)s * (COMP ? 2 : 1);
    double hi[kFixChains<COMP>], lo[kFixChains<COMP>];
#pragma unroll
    for (int j = 0; j < kFixChains<COMP>; j++) hi[j] = lo[j] = 0.0;
    // chain j takes units u + j * L: full rounds of kFixChains loads, then
    // one round of kFixChains, half or a quarter of them, whichever covers
    // the units left.  Its chains past nu read unit l again and add 0: no
    // branch, so a round's loads are all in flight together (a branch per
    // chain serialised them: R-MAT scale 22 s = 256 with 128-row slices,
    // SpMV 504 -> 584 us).
    constexpr int C = kFixChains<COMP>;
    uint32_t u = l;
    for (; u + (uint32_t)(C - 1) * L < nu; u += (uint32_t)C * L)
        fix_round<COMP, C>(part, stride, u0, u, l, L, nu, s, r, hi, lo);
    if (u < nu) {
        const uint32_t left = (nu - u + L - 1) / L;  // 1 .. C - 1
        if (left > (uint32_t)C / 2) fix_round<COMP, C>(part, stride, u0, u, l, L, nu, s, r, hi, lo);
        else if (left > (uint32_t)C / 4) fix_round<COMP, C / 2>(part, stride, u0, u, l, L, nu, s, r, hi, lo);
        else fix_round<COMP, C / 4>(part, stride, u0, u, l, L, nu, s, r, hi, lo);
    }
#pragma unroll
    for (int j = 1; j < kFixChains<COMP>; j++) fix_add<COMP>(hi[0], lo[0], hi[j], lo[j]);
    sh[threadIdx.x] = hi[0];
    if constexpr (COMP) sh[kFixThreads + threadIdx.x] = lo[0];
    __syncthreads();
    if (l == 0) {
        const uint32_t lr = (uint32_t)(r - r0);
        double H = 0.0, Lo = 0.0;
        for (uint32_t t = 0; t < L; t++)
            fix_add<COMP>(H, Lo, sh[t * (uint32_t)rs + lr], COMP ? sh[kFixThreads + t * (uint32_t)rs + lr] : 0.0);
        const int64_t gr = I * s + r;
        if (gr < m) {
            const double a = H + Lo;
            y[gr] = (beta == 0.0) ? alpha * a : alpha * a + beta * y[gr];
        }
    }
}

// Heavy strips of every matrix: hv[2h] = matrix, hv[2h+1] = heavy index.
// TIMED: thread 0 adds the workgroup's cycles times its wave count.
template <bool TIMED>
__global__ __launch_bounds__(kFixThreads) void k_batch_fixup(const BatchEntry *__restrict__ E,
                                                             const uint32_t *__restrict__ hv, double alpha,
                                                             double beta, unsigned long long *cyc)
{
    __shared__ double sh[2 * kFixThreads];
    long long t0 = 0;
    if constexpr (TIMED) t0 = clock64();
    const uint32_t mat = hv[2 * blockIdx.x];
    const BatchEntry &e = E[mat];
    const uint32_t h = hv[2 * blockIdx.x + 1];
    if (e.comp)  // workgroup-uniform
        fixup_strip<true>(e.A.s, e.A.s, 0, e.A.m, e.B.heavy[h * 3], e.B.part, e.B.heavy[h * 3 + 1],
                          e.B.heavy[h * 3 + 2], e.y, alpha, beta, sh);
    else
        fixup_strip<false>(e.A.s, e.A.s, 0, e.A.m, e.B.heavy[h * 3], e.B.part, e.B.heavy[h * 3 + 1],
                           e.B.heavy[h * 3 + 2], e.y, alpha, beta, sh);
    if constexpr (TIMED) {
        __syncthreads();
        if (threadIdx.x == 0)
            atomicAdd(&cyc[mat], (unsigned long long)(clock64() - t0) * (unsigned long long)(kFixThreads / kWave));
    }
}

// Rows of heavy strips (one workgroup per heavy strip).
template <bool COMP>
__global__ __launch_bounds__(kFixThreads) void k_spmv_fixup(int s, int64_t m, double *__restrict__ y, double alpha,
                                                            double beta, Balance B)
{
    __shared__ double sh[kFixThreads * (COMP ? 2 : 1)];
    // workgroup b sums rows [r0, r0 + rs) of heavy strip h (fix_rows)
    const uint32_t h = B.fix[2 * (size_t)blockIdx.x], w = B.fix[2 * (size_t)blockIdx.x + 1];
    const int r0 = (int)(w & 0xFFFFu), rs = (int)(w >> 16);
    fixup_strip<COMP>(s, rs, r0, m, B.heavy[h * 3], B.part, B.heavy[h * 3 + 1], B.heavy[h * 3 + 2], y, alpha, beta,
                      sh);
}

// LDS bytes per wave of the SpMM kernel: the s x R accumulator (twice when
// compensated), the decoded COO window (value, row, column) and the chunk's
// prefix sums and block columns.
__host__ __device__ inline size_t spmm_wave_lds(int s, int R, bool comp)
{
    return (size_t)s * R * sizeof(double) * (comp ? 2 : 1) + kWave * (sizeof(double) + 4 * sizeof(uint32_t));
}

// ===========================================================================
// Several right-hand sides (SpMM), R lanes per entry.
// ===========================================================================
// Dense s x s block times an s x R slice of X on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64: A 16x4 with lane l holding A[l%16][l/16], B 4x16
// with lane l holding B[l/16][l%16], D 16x16 with register r of lane l
// holding D[4r + l/16][l%16], r = 0..3; layout measured on gfx950).  The 16 x 16 product tiles are added to the
// strip accumulator (one lane per element, so no atomics).
template <typename VT, int R>
__device__ inline void dense_block_mfma(const VT *__restrict__ D, int s, int64_t c0, int64_t n,
                                        const double *__restrict__ X, int64_t ldx, int nrhs, double *acc, int lane)
{
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll 1
    for (int r0 = 0; r0 < s; r0 += 16) {
#pragma unroll
        for (int j0 = 0; j0 < R; j0 += 16) {
            typedef double v4d __attribute__((ext_vector_type(4)));
            v4d c = {0.0, 0.0, 0.0, 0.0};
            const int j = j0 + li;
#pragma unroll 4
            for (int k0 = 0; k0 < s; k0 += 4) {
                const double a = (double)D[(int64_t)(r0 + li) * s + k0 + lk];
                const int64_t gc = c0 + k0 + lk;
                const double bx = (gc < n && j < nrhs) ? X[gc * ldx + j] : 0.0;
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bx, c, 0, 0, 0);
            }
            // v_mfma_f64_16x16x4f64 result: register r of lane l holds row 4r + l/16, column l%16
            acc[(r0 + lk) * R + j] += c[0];
            acc[(r0 + 4 + lk) * R + j] += c[1];
            acc[(r0 + 8 + lk) * R + j] += c[2];
            acc[(r0 + 12 + lk) * R + j] += c[3];
        }
    }
}

// CSR group of the SpMM kernel, strip I.  Lanes own block rows as in the
// single-vector CSR walk (for s <= 64, lane l takes row l % s of block l / s
// of each step; for s > 64, one block per step in s / 64 row passes) and hold
// the row's R right-hand sides in registers: each entry's column and value
// are loaded once and its R values of X are read back to back (16-byte loads
// where X allows).  Row sums carry over the strip's blocks; the G = 64 / s
// lanes that share a row (s < 64) are summed with xor-shuffles, and the row's
// owner adds the sums to the accumulator (one writer per element: no atomics).
// X holds the wave's R columns (nrhs of them valid) at stride ldx.
// 27-point stencil 160^3, s = 64, FP64, k = 8 / k = 32: 1.10 / 4.07 ms, against
// 1.39 / 4.94 ms for a walk of 8 rows of R lanes per step (s * R / 64 chains
// of dependent loads per block).  More loads in flight per lane were slower
// throughout: two blocks per lane 1.43 / 5.87 ms, 2 or 4 entries per chain
// 1.38 / 5.10 and 1.62 / 6.04 ms, the next block's row pointers prefetched
// 1.22 / 4.52 ms -- the X reads queue in the memory pipeline (address unit
// busy 65 % of the time), not in each wave's dependency chain.
template <typename VT, typename BT, typename RT, int R, bool COMP>
__device__ inline void spmm_csr_rows(const DevMat &A, int64_t I, const double *__restrict__ X, int64_t ldx,
                                     int nrhs, const Acc &acc, uint32_t *s_st, uint32_t *s_bc, int lane)
{
    const uint32_t b0 = A.sptr[CSR][I], b1 = A.sptr[CSR][I + 1];
    if (b0 >= b1) return;
    uint32_t e = A.eptr[CSR][I];
    const int s = A.s;
    const int sw = s < kWave ? s : kWave;  // lanes per block
    const int G = kWave / sw;              // blocks per wave step
    const int passes = s / sw;             // row passes per block
    const int lb = lane / sw, lr = lane % sw;
    const int nr = nrhs < R ? nrhs : R;
    // whole tile, X rows 16-byte aligned: R / 2 double2 loads per entry
    const bool vec = nr == R && ((reinterpret_cast<uintptr_t>(X) & 15u) == 0) && ((ldx & 1) == 0);
    const VT *__restrict__ val = static_cast<const VT *>(A.val[CSR]);
    const uint8_t *__restrict__ ccol = A.csr_col;
    const RT *__restrict__ rowptr = static_cast<const RT *>(A.csr_rowptr);
#pragma unroll 1
    for (uint32_t cb = b0; cb < b1; cb += kWave) {
        const uint32_t jb = cb + lane;
        const bool ok = jb < b1;
        const uint32_t z = ok ? (uint32_t)A.z1[CSR][jb] + 1u : 0u;
        const uint32_t incl = wave_incl_scan_dpp(z);
        s_st[lane] = e + incl - z;
        s_bc[lane] = ok ? (uint32_t)ld<BT>(A.bcol[CSR], jb) : 0u;
        e += (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        wave_sync();
        const int nbk = (int)min<uint32_t>(kWave, b1 - cb);
#pragma unroll 1
        for (int ps = 0; ps < passes; ps++) {
            const int r = ps * sw + lr;
            double hi[R], lo[R];
#pragma unroll
            for (int jj = 0; jj < R; jj++) hi[jj] = lo[jj] = 0.0;
#pragma unroll 1
            for (int j0 = 0; j0 < nbk; j0 += G) {
                const int jblk = j0 + lb;
                const bool h = jblk < nbk;
                const RT *rp = rowptr + (uint64_t)(cb + (uint32_t)(h ? jblk : 0)) * (uint64_t)(s + 1);
                const uint32_t ra = h ? (uint32_t)rp[r] : 0u, rc = h ? (uint32_t)rp[r + 1] : 0u;
                const uint32_t q0 = h ? s_st[jblk] + ra : 0u, ql = rc - ra;
                const int64_t xc = h ? (int64_t)s_bc[jblk] * s : 0;
                // (the loads below carry the t < ql predicate although it holds
                // inside the loop: that form measured 5 % faster, k = 32 4.07
                // against 4.27 ms)
                const uint32_t len = max(0u, ql);
#pragma unroll 1
                for (uint32_t t = 0; t < len; t++) {
                    double v, xv[R];
                    int64_t xr;
                    const bool hh = t < ql;
                    xr = hh ? (xc + ccol[q0 + t]) * ldx : 0;
                    v = hh ? (double)val[q0 + t] : 0.0;
                    bool done = false;
                    if constexpr (R >= 2) {
                        if (vec) {  // 16-byte loads: half the address work per value
                            const double2 *xp = reinterpret_cast<const double2 *>(X + xr);
#pragma unroll
                            for (int jj = 0; jj < R; jj += 2) {
                                double2 w = {0.0, 0.0};
                                if (hh) w = xp[jj >> 1];
                                xv[jj] = w.x;
                                xv[jj + 1] = w.y;
                            }
                            done = true;
                        }
                    }
                    if (!done) {
#pragma unroll
                        for (int jj = 0; jj < R; jj++) xv[jj] = (hh && jj < nr) ? X[xr + jj] : 0.0;
                    }
                    if (hh) {
#pragma unroll
                        for (int jj = 0; jj < R; jj++) acc_add<COMP>(hi[jj], lo[jj], v, xv[jj]);
                    }
                }
            }
            for (int o = sw; o < kWave; o <<= 1) {
#pragma unroll
                for (int jj = 0; jj < R; jj++) {
                    const double q = __shfl_xor(hi[jj], o, kWave);
                    if constexpr (COMP) {
                        const double qe = __shfl_xor(lo[jj], o, kWave);
                        double sum, err;
                        two_sum(hi[jj], q, sum, err);
                        hi[jj] = sum;
                        lo[jj] += qe + err;
                    } else {
                        hi[jj] += q;
                    }
                }
            }
            if (lb == 0) {
#pragma unroll
                for (int jj = 0; jj < R; jj++) {
                    if (jj >= nr) break;
                    const uint32_t ai = (uint32_t)r * R + jj;
                    if constexpr (COMP) {
                        double sum, err;
                        two_sum(acc.hi[ai], hi[jj], sum, err);
                        acc.hi[ai] = sum;
                        acc.lo[ai] += err + lo[jj];
                    } else {
                        acc.hi[ai] += hi[jj];
                    }
                }
            }
        }
        wave_sync();
    }
}

// Products of a decoded window of nq <= 64 entries (rows d_row, X rows
// d_col, values d_val, in LDS) with the wave's R columns of X, added to the
// strip accumulator with LDS atomics.  With a whole, 16-byte aligned tile
// (vec) H = R / 2 lanes take an entry, a double2 of X each, so H steps of
// 64 / H entries cover the window and all of its X loads are issued before
// its adds (one memory round trip per window; R-lane steps of one column per
// lane, below, wait for each step's loads in turn).
template <int R, bool COMP>
__device__ inline void spmm_window(uint32_t nq, const uint32_t *d_row, const uint32_t *d_col, const double *d_val,
                                   const double *__restrict__ X, int64_t ldx, int nrhs, bool vec, const Acc &acc,
                                   int lane)
{
    if constexpr (R >= 2) {
        if (vec) {
            constexpr int H = R / 2, E2 = kWave / H;
            const int slot2 = lane / H, c2 = lane % H;
            double2 xw[H];
#pragma unroll
            for (int g = 0; g < H; g++) {
                const uint32_t ent = (uint32_t)(g * E2 + slot2);
                xw[g] = double2{0.0, 0.0};
                if (ent < nq) xw[g] = reinterpret_cast<const double2 *>(X + (int64_t)d_col[ent] * ldx)[c2];
            }
            if constexpr (COMP) {
                // every returning add of the window first, then the TwoSums and
                // the compensation adds: the hi and lo arrays each receive their
                // adds in the same order as one product at a time, so the sums
                // are the same, but the returns are awaited once
                double p[2 * H], pe[2 * H], old[2 * H];
                uint32_t ai[2 * H];
#pragma unroll
                for (int g = 0; g < H; g++) {
                    const uint32_t ent = (uint32_t)(g * E2 + slot2);
                    const bool ok = ent < nq;
                    const double v = ok ? d_val[ent] : 0.0;
                    ai[2 * g] = ok ? d_row[ent] * R + 2 * c2 : 0u;
                    ai[2 * g + 1] = ai[2 * g] + 1;
                    p[2 * g] = prod<true>(v, xw[g].x, pe[2 * g]);
                    p[2 * g + 1] = prod<true>(v, xw[g].y, pe[2 * g + 1]);
                }
#pragma unroll
                for (int i = 0; i < 2 * H; i++)
                    if ((uint32_t)((i >> 1) * E2 + slot2) < nq) old[i] = atomicAdd(&acc.hi[ai[i]], p[i]);
#pragma unroll
                for (int i = 0; i < 2 * H; i++)
                    if ((uint32_t)((i >> 1) * E2 + slot2) < nq) {
                        double sum, err;
                        two_sum(old[i], p[i], sum, err);
                        atomicAdd(&acc.lo[ai[i]], err + pe[i]);
                    }
                return;
            }
#pragma unroll
            for (int g = 0; g < H; g++) {
                const uint32_t ent = (uint32_t)(g * E2 + slot2);
                if (ent < nq) {
                    const double v = d_val[ent];
                    const uint32_t ai = d_row[ent] * R + 2 * c2;
                    double pe;
                    double p = prod<COMP>(v, xw[g].x, pe);
                    acc_atomic<COMP>(acc, ai, p, pe);
                    p = prod<COMP>(v, xw[g].y, pe);
                    acc_atomic<COMP>(acc, ai + 1, p, pe);
                }
            }
            return;
        }
    }
    constexpr int E = kWave / R;  // entries per step
    const int slot = lane / R, j = lane % R;
#pragma unroll 1
    for (uint32_t g = 0; g < nq; g += E) {
        const uint32_t ent = g + slot;
        if (ent < nq && j < nrhs) {
            const double xv = X[(int64_t)d_col[ent] * ldx + j];
            double pe;
            const double p = prod<COMP>(d_val[ent], xv, pe);
            acc_atomic<COMP>(acc, d_row[ent] * R + j, p, pe);
        }
    }
}

// Two launch shapes: sib == 0, wave w of workgroup b takes strip b * wpb + w
// for the R right-hand sides at X, Y; sib > 0, the workgroup's sib waves all
// take strip b, wave w the R-column tile w of the sib * R columns (nrhs in
// all): the siblings read the same matrix entries together, so the matrix
// streams from HBM once for all tiles and the tiles' X values share cache
// lines in the CU's L1.
template <typename VT, typename BT, typename IT, typename RT, int R, bool COMP>
__global__ __launch_bounds__(256) void k_spmm_strip(DevMat A, const double *__restrict__ X, int64_t ldx,
                                                    double *__restrict__ Y, int64_t ldy, int nrhs,
                                                    double alpha, double beta, int wpb, int64_t nstrip_total,
                                                    int sib)
{
    constexpr int E = kWave / R;  // entries per wave step
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int slot = lane / R, j = lane % R;
    const int s = A.s, k = A.k;
    int64_t I = (int64_t)blockIdx.x * wpb + wave;
    if (sib) {
        I = blockIdx.x;
        X += (int64_t)wave * R;
        Y += (int64_t)wave * R;
        nrhs -= wave * R;
        if (nrhs <= 0) return;  // whole wave leaves; no workgroup barriers below
    }
    const bool jok = j < nrhs;
    if (I >= nstrip_total) return;  // whole wave leaves; no workgroup barriers below
    // whole tile, X rows 16-byte aligned: the decoded windows read X as double2
    const bool vec = nrhs >= R && ((reinterpret_cast<uintptr_t>(X) & 15u) == 0) && ((ldx & 1) == 0);

    const size_t per_wave = spmm_wave_lds(s, R, COMP);
    unsigned char *base = smem + per_wave * wave;
    Acc acc;
    acc.hi = reinterpret_cast<double *>(base);
    acc.lo = COMP ? acc.hi + (size_t)s * R : nullptr;
    double *d_val = reinterpret_cast<double *>(base + (size_t)s * R * sizeof(double) * (COMP ? 2 : 1));
    uint32_t *s_end = reinterpret_cast<uint32_t *>(d_val + kWave);
    uint32_t *s_bc = s_end + kWave;
    uint32_t *d_row = s_bc + kWave;
    uint32_t *d_col = d_row + kWave;

    for (int i = lane; i < s * R; i += kWave) {
        acc.hi[i] = 0.0;
        if constexpr (COMP) acc.lo[i] = 0.0;
    }
    wave_sync();

    const uint32_t smask = (uint32_t)s - 1;

    // ---- COO group: windows of 64 entries are decoded once (one entry per
    // lane: block by binary search over the chunk's prefix sums, local row and
    // global column, value) into LDS, then E = 64/R entries per step times R
    // right-hand sides read the decoded window -------------------------------
    {
        const uint32_t b0 = A.sptr[COO][I], b1 = A.sptr[COO][I + 1];
        uint32_t e = A.eptr[COO][I];
        const VT *val = static_cast<const VT *>(A.val[COO]);
#pragma unroll 1
        for (uint32_t cb = b0; cb < b1; cb += kWave) {
            const uint32_t jb = cb + lane;
            const bool ok = jb < b1;
            const uint32_t z = ok ? (uint32_t)A.z1[COO][jb] + 1u : 0u;
            const uint32_t incl = wave_incl_scan_dpp(z);
            const uint32_t T = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
            s_end[lane] = incl;
            s_bc[lane] = ok ? (uint32_t)ld<BT>(A.bcol[COO], jb) : 0u;
            wave_sync();
            const int nbk = (int)min<uint32_t>(kWave, b1 - cb);
#pragma unroll 1
            for (uint32_t q = 0; q < T; q += kWave) {
                const uint32_t t = q + lane;
                if (t < T) {
                    int lo = 0, hi = nbk - 1;  // first chunk block with end > t
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (s_end[mid] > t) hi = mid; else lo = mid + 1;
                    }
                    const uint32_t id = ld<IT>(A.coo_idx, e + t);
                    d_row[lane] = id >> k;
                    d_col[lane] = s_bc[lo] * (uint32_t)s + (id & smask);
                    d_val[lane] = (double)val[e + t];
                }
                wave_sync();
                spmm_window<R, COMP>(min<uint32_t>(kWave, T - q), d_row, d_col, d_val, X, ldx, nrhs, vec, acc, lane);
                wave_sync();
            }
            e += T;
        }
    }

    // ---- CSR group: lanes own block rows, R right-hand sides per lane in
    // registers across the strip's blocks
    spmm_csr_rows<VT, BT, RT, R, COMP>(A, I, X, ldx, nrhs, acc, s_end, s_bc, lane);
    // ---- bitmap and dense groups: position-parallel over 64-bit words --------
    // Within a word, positions t*E + slot (t < R) share a row in aligned groups
    // of G = min(E, s) slots, so products are summed with xor-shuffles over the
    // slot bits and the group leader updates the row (no two leaders of one
    // step hit the same row and rhs, so no atomics are needed).
    const int G = E < s ? E : s;
    const int W = A.W;
    const uint32_t ssq = (uint32_t)s * (uint32_t)s;
#pragma unroll 1
    for (int sc = BITMAP; sc <= DENSE; sc++) {
        const uint32_t b0 = A.sptr[sc][I], b1 = A.sptr[sc][I + 1];
        uint64_t vbase = (sc == BITMAP) ? (uint64_t)A.eptr[BITMAP][I] : 0;
        const VT *val = static_cast<const VT *>(A.val[sc]);
#pragma unroll 1
        for (uint32_t b = b0; b < b1; b++) {
            const int64_t c0 = (int64_t)ld<BT>(A.bcol[sc], b) * s;
            const uint64_t *words = A.bm_words + (uint64_t)b * W;
            if (sc == DENSE) vbase = (uint64_t)b * ssq;
            if constexpr (R >= 16 && !COMP) {
                if (sc == DENSE && s >= 16) {
                    dense_block_mfma<VT, R>(val + vbase, s, c0, A.n, X, ldx, nrhs, acc.hi, lane);
                    continue;
                }
            }
            if constexpr (R >= 2) {
                if (sc == BITMAP) {
                    // decode each word's set bits (in value order) into the
                    // window, then E entries x R right-hand sides per step:
                    // no step is spent on empty positions
#pragma unroll 1
                    for (int w = 0; w < W; w++) {
                        const uint64_t word = words[w];
                        const uint32_t nq = (uint32_t)__popcll(word);
                        if ((word >> lane) & 1ull) {
                            const uint32_t ix = (uint32_t)__popcll(word & ((1ull << lane) - 1ull));
                            const uint32_t pos = (uint32_t)w * 64u + (uint32_t)lane;
                            d_row[ix] = pos >> k;
                            d_col[ix] = (uint32_t)(c0 + (pos & smask));
                            d_val[ix] = (double)val[vbase + ix];
                        }
                        wave_sync();
                        spmm_window<R, COMP>(nq, d_row, d_col, d_val, X, ldx, nrhs, vec, acc, lane);
                        wave_sync();
                        vbase += nq;
                    }
                    continue;
                }
            }
#pragma unroll 1
            for (int w = 0; w < W; w++) {
                const uint64_t word = (sc == BITMAP) ? words[w] : ~0ull;
                for (int t = 0; t < R; t++) {
                    const uint32_t i = (uint32_t)(t * E + slot);  // bit within the word
                    const uint32_t pos = (uint32_t)w * 64u + i;    // position in the block
                    const bool inb = pos < ssq;
                    const bool bit = inb && ((word >> i) & 1ull);
                    const uint32_t lr = pos >> k, lc = pos & smask;
                    double p = 0.0, pe = 0.0;
                    if (bit && jok) {
                        const uint64_t vi = (sc == BITMAP) ? vbase + __popcll(word & ((1ull << i) - 1ull))
                                                           : vbase + pos;
                        const int64_t gc = c0 + lc;
                        const double xv = (gc < A.n) ? X[gc * ldx + j] : 0.0;
                        p = prod<COMP>((double)val[vi], xv, pe);
                    }
                    for (int o = (G >> 1) * R; o >= R; o >>= 1) {
                        const double q = __shfl_xor(p, o, kWave);
                        if constexpr (COMP) {
                            const double qe = __shfl_xor(pe, o, kWave);
                            double sum, err;
                            two_sum(p, q, sum, err);
                            p = sum;
                            pe += qe + err;
                        } else {
                            p += q;
                        }
                    }
                    if ((slot & (G - 1)) == 0 && inb && jok) {
                        const uint32_t ai = lr * R + j;
                        if constexpr (COMP) {
                            double sum, err;
                            two_sum(acc.hi[ai], p, sum, err);
                            acc.hi[ai] = sum;
                            acc.lo[ai] += err + pe;
                        } else {
                            acc.hi[ai] += p;
                        }
                    }
                }
                wave_sync();
                if (sc == BITMAP) vbase += __popcll(word);  // dense positions are absolute
            }
        }
    }

    wave_sync();
    // ---- write the strip's rows ---------------------------------------------
    for (int i = lane; i < s * R; i += kWave) {
        const int r = i / R, jj = i % R;
        const int64_t gr = I * s + r;
        if (gr >= A.m || jj >= nrhs) continue;
        double a = acc.hi[i];
        if constexpr (COMP) a += acc.lo[i];
        double *yp = Y + gr * ldy + jj;
        *yp = (beta == 0.0) ? alpha * a : alpha * a + beta * *yp;
    }
}

// nrhs <= R: one tile, wpb strips per workgroup; nrhs > R (at most
// kSpmmSiblings * R): sibling waves, one strip per workgroup, one R-column
// tile per wave.
constexpr int kSpmmSiblings = 4;

template <typename VT, typename BT, typename IT, typename RT, int R, bool COMP>
void launch_t(const DevMat &A, const double *X, int64_t ldx, double *Y, int64_t ldy, int nrhs, double alpha,
              double beta, hipStream_t st)
{
    const size_t per_wave = spmm_wave_lds(A.s, R, COMP);
    const int sib = nrhs > R ? (nrhs + R - 1) / R : 0;
    ABHSF_REQUIRE(sib <= kSpmmSiblings, ABHSF_ERR_UNSUPPORTED, "more column tiles than sibling waves");
    int wpb = sib ? sib : (int)(65536 / per_wave);
    if (wpb > 4) wpb = 4;
    ABHSF_REQUIRE(wpb >= 1 && per_wave * wpb <= 65536, ABHSF_ERR_UNSUPPORTED, "output tile does not fit in LDS");
    const int64_t nblk = sib ? A.M : (A.M + wpb - 1) / wpb;
    ABHSF_REQUIRE(nblk < (1ll << 31), ABHSF_ERR_UNSUPPORTED, "too many strips");
    if (A.M == 0) return;
    hipLaunchKernelGGL((k_spmm_strip<VT, BT, IT, RT, R, COMP>), dim3((unsigned)nblk), dim3(64 * wpb),
                       per_wave * wpb, st, A, X, ldx, Y, ldy, nrhs, alpha, beta, wpb, A.M, sib);
    ABHSF_HIP(hipGetLastError());
}

template <typename VT, typename BT, typename IT, typename RT, bool COMP>
void launch_spmv(const DevMat &A, const Balance &B, const double *x, double *y, double alpha,
                 double beta, hipStream_t st)
{
    if (A.M == 0) return;
    Balance b = B;
    if (!b.light && b.n_units == 0) b.n_light = A.M;  // one item per strip
    const int64_t nitems = b.n_light + b.n_units;
    const int64_t nblk = b.order ? b.n_slots / kStripWaves : (nitems + kStripWaves - 1) / kStripWaves;
    ABHSF_REQUIRE(nblk < (1ll << 31), ABHSF_ERR_UNSUPPORTED, "too many strips");
    // tiled matrices have their own kernels (each carries one light-item
    // path); the choice is made once, here: a tiled storage read by an untiled
    // kernel would take its z1 strip bits for entry counts
    const StripArgs args{A, b, x, y, alpha, beta};
    if (b.tiled)
        hipLaunchKernelGGL((k_spmv_strip<VT, BT, IT, RT, COMP, true>), dim3((unsigned)nblk), dim3(64 * kStripWaves), 0,
                           st, args);
    else
        hipLaunchKernelGGL((k_spmv_strip<VT, BT, IT, RT, COMP, false>), dim3((unsigned)nblk), dim3(64 * kStripWaves),
                           0, st, args);
    ABHSF_HIP(hipGetLastError());
    if (b.n_heavy) {
        ABHSF_REQUIRE(b.n_fix > 0 && b.n_fix < (1ll << 31), ABHSF_ERR_STATE, "fix-up table missing");
        hipLaunchKernelGGL((k_spmv_fixup<COMP>), dim3((unsigned)b.n_fix), dim3(kFixThreads), 0, st, A.s, A.m, y,
                           alpha, beta, b);
        ABHSF_HIP(hipGetLastError());
    }
}

template <typename VT, typename BT, typename IT, typename RT, bool COMP>
void launch_r(int R, const DevMat &A, const Balance &Bal, const double *X, int64_t ldx, double *Y,
              int64_t ldy, int nrhs, double alpha, double beta, hipStream_t st)
{
    switch (R) {
    case 1:
        if (nrhs == 1 && ldx == 1 && ldy == 1)
            launch_spmv<VT, BT, IT, RT, COMP>(A, Bal, X, Y, alpha, beta, st);
        else launch_t<VT, BT, IT, RT, 1, COMP>(A, X, ldx, Y, ldy, nrhs, alpha, beta, st);
        break;
    case 2: launch_t<VT, BT, IT, RT, 2, COMP>(A, X, ldx, Y, ldy, nrhs, alpha, beta, st); break;
    case 4: launch_t<VT, BT, IT, RT, 4, COMP>(A, X, ldx, Y, ldy, nrhs, alpha, beta, st); break;
    case 8: launch_t<VT, BT, IT, RT, 8, COMP>(A, X, ldx, Y, ldy, nrhs, alpha, beta, st); break;
    case 16: launch_t<VT, BT, IT, RT, 16, COMP>(A, X, ldx, Y, ldy, nrhs, alpha, beta, st); break;
    case 32: launch_t<VT, BT, IT, RT, 32, COMP>(A, X, ldx, Y, ldy, nrhs, alpha, beta, st); break;
    default: throw Error(ABHSF_ERR_UNSUPPORTED, "unsupported rhs tile");
    }
}

template <typename VT, bool COMP>
void launch_v(const SpmvLaunch &L, const DevMat &A, int R, const double *X, int64_t ldx, double *Y, int64_t ldy,
              int nrhs, double alpha, double beta, hipStream_t st)
{
    const Balance &Bal = L.bal;
    const bool b16 = L.bcol_bytes == 2;
    const int s = A.s;
    if (s <= 8) {
        if (b16) launch_r<VT, uint16_t, uint8_t, uint8_t, COMP>(R, A, Bal, X, ldx, Y, ldy, nrhs, alpha, beta, st);
        else launch_r<VT, uint32_t, uint8_t, uint8_t, COMP>(R, A, Bal, X, ldx, Y, ldy, nrhs, alpha, beta, st);
    } else if (s <= 16) {
        if (b16) launch_r<VT, uint16_t, uint8_t, uint16_t, COMP>(R, A, Bal, X, ldx, Y, ldy, nrhs, alpha, beta, st);
        else launch_r<VT, uint32_t, uint8_t, uint16_t, COMP>(R, A, Bal, X, ldx, Y, ldy, nrhs, alpha, beta, st);
    } else {
        if (b16) launch_r<VT, uint16_t, uint16_t, uint16_t, COMP>(R, A, Bal, X, ldx, Y, ldy, nrhs, alpha, beta, st);
        else launch_r<VT, uint32_t, uint16_t, uint16_t, COMP>(R, A, Bal, X, ldx, Y, ldy, nrhs, alpha, beta, st);
    }
}

}  // namespace

int fix_rows(int s, uint32_t nu, bool comp)
{
    int rs = std::min(s, comp ? kFixRows<true> : kFixRows<false>);
    while (rs > kFixRowsMin && (uint64_t)nu * (uint64_t)rs > (uint64_t)kFixUnits * (uint64_t)kFixThreads) rs /= 2;
    return rs;
}

int batch_code(int bcol_bytes, int s) { return (bcol_bytes == 4 ? 3 : 0) + (s <= 8 ? 0 : (s <= 16 ? 1 : 2)); }

void batch_spmv(const BatchEntry *dE, const uint32_t *item_mat, int64_t G64, int64_t G, const uint32_t *dheavy,
                int64_t nheavy, double alpha, double beta, hipStream_t st, unsigned long long *cycles)
{
    auto launch = [&](auto comp_tag, int64_t g0, int64_t g1) {
        constexpr bool C = decltype(comp_tag)::value;
        if (g1 <= g0) return;
        const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((g1 - g0 + 3) / 4, 8192));
        if (cycles)
            hipLaunchKernelGGL((k_batch_spmv<true, C>), dim3((unsigned)grid), dim3(256), 0, st, dE, item_mat, g0, g1,
                               alpha, beta, cycles);
        else
            hipLaunchKernelGGL((k_batch_spmv<false, C>), dim3((unsigned)grid), dim3(256), 0, st, dE, item_mat, g0,
                               g1, alpha, beta, cycles);
        ABHSF_HIP(hipGetLastError());
    };
    launch(std::integral_constant<bool, false>{}, 0, G64);
    launch(std::integral_constant<bool, true>{}, G64, G);
    if (nheavy > 0) {
        if (cycles)
            hipLaunchKernelGGL(k_batch_fixup<true>, dim3((unsigned)nheavy), dim3(kFixThreads), 0, st, dE, dheavy,
                               alpha, beta, cycles);
        else
            hipLaunchKernelGGL(k_batch_fixup<false>, dim3((unsigned)nheavy), dim3(kFixThreads), 0, st, dE, dheavy,
                               alpha, beta, cycles);
        ABHSF_HIP(hipGetLastError());
    }
}

void spmv_transposed(const SpmvLaunch &L, const DevMat &A, int nrhs, double scale, const double *X, int64_t ldx,
                     double *Y, int64_t ldy, hipStream_t st)
{
    ABHSF_REQUIRE(L.val_bytes == 8, ABHSF_ERR_UNSUPPORTED, "symmetric storage needs FP64 values");
    if (A.M == 0) return;
    Balance b = L.bal;
    if (!b.light && b.n_units == 0) b.n_lstrips = A.M;
    const int64_t nblk = (b.n_lstrips + b.n_units + kStripWaves - 1) / kStripWaves;
    ABHSF_REQUIRE(nblk < (1ll << 31), ABHSF_ERR_UNSUPPORTED, "too many strips");
    const bool b16 = L.bcol_bytes == 2;
    for (int j = 0; j < nrhs; j++) {
        const TransArgs args{A, b, X + j, Y + j, ldx, ldy, scale};
#define ABHSF_TRANS(BT_, IT_, RT_) \
    hipLaunchKernelGGL((k_spmv_trans<BT_, IT_, RT_>), dim3((unsigned)nblk), dim3(64 * kStripWaves), 0, st, args)
        if (A.s <= 8) {
            if (b16) ABHSF_TRANS(uint16_t, uint8_t, uint8_t); else ABHSF_TRANS(uint32_t, uint8_t, uint8_t);
        } else if (A.s <= 16) {
            if (b16) ABHSF_TRANS(uint16_t, uint8_t, uint16_t); else ABHSF_TRANS(uint32_t, uint8_t, uint16_t);
        } else {
            if (b16) ABHSF_TRANS(uint16_t, uint16_t, uint16_t); else ABHSF_TRANS(uint32_t, uint16_t, uint16_t);
        }
#undef ABHSF_TRANS
        ABHSF_HIP(hipGetLastError());
    }
}

namespace {
// Column blocks between a row-major n x ld array and contiguous columns
// (column c of the block at dst + c * rows), through a transposed LDS tile so
// that both sides are read and written in whole rows / runs: a workgroup
// takes 256 rows of at most kColBlock columns.
constexpr int kColBlock = 8;

__global__ __launch_bounds__(256) void k_gather_cols(const double *__restrict__ src, int64_t lds, int64_t rows,
                                                     int cols, double *__restrict__ dst)
{
    __shared__ double t[kColBlock][257];
    const int64_t r0 = (int64_t)blockIdx.x * 256;
    for (int e = threadIdx.x; e < 256 * cols; e += 256) {
        const int rr = e / cols, c = e % cols;
        if (r0 + rr < rows) t[c][rr] = src[(r0 + rr) * lds + c];
    }
    __syncthreads();
    const int64_t r = r0 + threadIdx.x;
    if (r < rows)
        for (int c = 0; c < cols; c++) dst[(int64_t)c * rows + r] = t[c][threadIdx.x];
}

__global__ __launch_bounds__(256) void k_scatter_cols(const double *__restrict__ src, int64_t rows, int cols,
                                                      double *__restrict__ dst, int64_t ldd)
{
    __shared__ double t[kColBlock][257];
    const int64_t r0 = (int64_t)blockIdx.x * 256;
    const int64_t r = r0 + threadIdx.x;
    if (r < rows)
        for (int c = 0; c < cols; c++) t[c][threadIdx.x] = src[(int64_t)c * rows + r];
    __syncthreads();
    for (int e = threadIdx.x; e < 256 * cols; e += 256) {
        const int rr = e / cols, c = e % cols;
        if (r0 + rr < rows) dst[(r0 + rr) * ldd + c] = t[c][rr];
    }
}
}  // namespace

int col_block() { return kColBlock; }

void gather_cols(const double *src, int64_t lds, int64_t rows, int cols, double *dst, hipStream_t st)
{
    ABHSF_REQUIRE(cols >= 1 && cols <= kColBlock, ABHSF_ERR_INVALID, "column block too wide");
    if (rows <= 0) return;
    const int64_t nblk = (rows + 255) / 256;
    ABHSF_REQUIRE(nblk < (1ll << 31), ABHSF_ERR_UNSUPPORTED, "vector too long");
    hipLaunchKernelGGL(k_gather_cols, dim3((unsigned)nblk), dim3(256), 0, st, src, lds, rows, cols, dst);
    ABHSF_HIP(hipGetLastError());
}

void scatter_cols(const double *src, int64_t rows, int cols, double *dst, int64_t ldd, hipStream_t st)
{
    ABHSF_REQUIRE(cols >= 1 && cols <= kColBlock, ABHSF_ERR_INVALID, "column block too wide");
    if (rows <= 0) return;
    const int64_t nblk = (rows + 255) / 256;
    ABHSF_REQUIRE(nblk < (1ll << 31), ABHSF_ERR_UNSUPPORTED, "vector too long");
    hipLaunchKernelGGL(k_scatter_cols, dim3((unsigned)nblk), dim3(256), 0, st, src, rows, cols, dst, ldd);
    ABHSF_HIP(hipGetLastError());
}

int max_rhs_tile(int s, bool comp)
{
    int R = 32;
    while (R > 1 && spmm_wave_lds(s, R, comp) > 65536) R >>= 1;
    return R;
}

void spmm(const SpmvLaunch &L, const DevMat &A, int nrhs, double alpha, const double *X, int64_t ldx, double beta,
          double *Y, int64_t ldy, hipStream_t st)
{
    const bool comp = L.val_bytes == 4;
    // column tiles of at most 8 right-hand sides (16 with dense blocks, whose
    // tiles go through the FP64 matrix cores from R = 16): wider tiles hold a
    // larger s x R accumulator in LDS per wave and lose more occupancy than
    // the extra pass over the matrix costs (stencil27, s = 64: k = 32 as one
    // tile 12.2 ms, as 2 x 16 4.3 ms each, as 4 x 8 1.5 ms each)
    // up to kSpmmSiblings tiles per launch go to sibling waves of one strip
    // (the matrix is read once for all of them)
    const int rmax = std::min(max_rhs_tile(A.s, comp), L.has_dense && !comp ? 16 : 8);
    const int sibmax = std::max(1, std::min(kSpmmSiblings, (int)(65536 / spmm_wave_lds(A.s, rmax, comp))));
    const int span = rmax * sibmax;
    for (int j0 = 0; j0 < nrhs; j0 += span) {
        const int nr = nrhs - j0 < span ? nrhs - j0 : span;
        int R = 1;
        while (R < nr && R < rmax) R <<= 1;
        if (comp) launch_v<float, true>(L, A, R, X + j0, ldx, Y + j0, ldy, nr, alpha, beta, st);
        else launch_v<double, false>(L, A, R, X + j0, ldx, Y + j0, ldy, nr, alpha, beta, st);
    }
}

}  // namespace abhsf
