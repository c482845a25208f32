// Shared pieces of the sparse kernels: deterministic grid reductions, the hybrid
// SELL-C-sigma device view and its row kernel, launch helpers and the SpMV timer.
#pragma once
#include <algorithm>
#include <string>
#include <hip/hip_ext.h>
#include "mk_internal.h"
#include <chrono>

namespace mk {

static constexpr int kMaxWaves = 16;        // 1024 threads / 64
static constexpr size_t kMaxParts = 1 << 17;  // partial-sum slots per reduced quantity
static constexpr int kMaxK = 4;
// Longest row kept in the SELL part; longer rows go to the medium (lane group per row) or
// long (wavefront per row) parts at upload, so SELL slice widths never exceed it.
static constexpr int kSellMaxLen = 12;
// Entries per segment of a long row in the multi-column kernels (a 1,330-entry row: 11
// wavefronts instead of one serial chain)
static constexpr int kLongSeg = 128;

// Sum over the wavefront, the same in every lane, by DPP row shifts and broadcasts: no LDS round
// trips (the xor-butterfly's twelve ds_bpermute per double made a reduction of 16 quantities take
// 4 us).  Fixed order.
template <int CTRL>
__device__ __forceinline__ double dpp_shift(double v) {  // lanes without a source get 0
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// row_bcast: the last lane of a row of 16 to the next row (CTRL 0x142, rows 1 and 3) or of the lower
// half to the upper (0x143, rows 2 and 3); other rows get 0
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_bcast(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_shift<0x111>(v);  // row_shr:1, 2, 4, 8
    v += dpp_shift<0x112>(v);
    v += dpp_shift<0x114>(v);
    v += dpp_shift<0x118>(v);
    v += dpp_bcast<0x142, 0xa>(v);
    v += dpp_bcast<0x143, 0xc>(v);
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Block-reduce K values; every thread gets the block totals.  One barrier: a kernel that reduces more
// than once gives each reduction its own TAG (its own LDS).
template <int K, int TAG = 0>
__device__ __forceinline__ void block_sum(double (&v)[K]) {
    __shared__ double sh[K][kMaxWaves];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const double s = wave_sum(v[k]);
        if (lane == 0) sh[k][wid] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; k++) {
        double s = 0.0;
        for (int w = 0; w < nw; w++) s += sh[k][w];
        v[k] = s;
    }
}

// Fence-free grid reduction in two launches: the working kernel leaves one partial sum per
// block (partials[k * kMaxParts + block]) and a one-block finishing kernel adds them in a fixed
// order after the kernel boundary.  No device-scope fence or ticket per block: on a chip whose
// L2 is private to each XCD a device-scope release writes back the block's L2, which costs far
// more than the extra launch in kernels that stream large vectors.
template <int K>
__device__ __forceinline__ void partials_write(double (&v)[K], double* partials) {
    block_sum<K>(v);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < K; k++) partials[k * kMaxParts + blockIdx.x] = v[k];
    }
}
// Sum of nparts partials per value, fixed order; every thread of the block gets tot.
template <int K>
__device__ __forceinline__ void partials_sum(const double* __restrict__ partials, int nparts, double (&tot)[K]) {
#pragma unroll
    for (int k = 0; k < K; k++) tot[k] = 0.0;
#pragma unroll 4
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
#pragma unroll
        for (int k = 0; k < K; k++) tot[k] += partials[k * kMaxParts + i];
    }
    block_sum<K, 1>(tot);
}

// Tells the host whether the start meets the tolerance (mk_ctx::started: page-locked memory).
__device__ __forceinline__ void tell_start(int* started, int done) {
    __hip_atomic_store(started, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The blocks of a launch go round-robin over the 8 XCDs, each with its own L2.  xcd_block maps
// the hardware block id b in [0, nb) to a logical block id so that every XCD works through one
// contiguous range of logical blocks: neighbouring rows then find the x entries they gather
// in their own XCD's L2.  A bijection for any nb.
static constexpr int kXcd = 8;
__device__ __forceinline__ int xcd_block(int b, int nb) {
    const int x = b % kXcd, q = nb / kXcd, r = nb % kXcd;
    return x * q + (x < r ? x : r) + b / kXcd;
}

template <typename T>
struct SellDev {
    int n_short, C, nb_sell, nlong;
    int nvb;  // virtual blocks: nb_sell SELL blocks, nb_mid medium-row blocks, then long-row blocks
    int nb_mid, nmid, mid_lanes;
    const int* mid_rows;
    const int64_t* mid_ptr;
    const int* mid_col;
    const T* mid_val;
    const int64_t* slice_ptr;
    const int* slice_w;
    const int* col;
    const T* val;
    const int* perm;
    const int* long_rows;
    const int64_t* long_ptr;
    const int* long_col;
    const T* long_val;
    int nseg;                // long-row segments (multi-column kernels)
    const int64_t* seg_beg;
    const int64_t* seg_end;
    const int* lseg_ptr;
    T* seg_part;
};

template <typename T>
__device__ __forceinline__ T wave_sum_t(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Vector access of the row kernels: a gather g(c, xr, xi) loads entry c of the vector the
// operator multiplies (xi unused for real operators).
template <typename T, bool CPLX>
struct PlainGather {
    const T* __restrict__ x;
    __device__ __forceinline__ void operator()(int c, T& xr, T& xi) const {
        if constexpr (CPLX) { xr = x[2 * c]; xi = x[2 * c + 1]; }
        else { xr = x[c]; xi = T(0); }
    }
};

// No row-local operands to fetch early.
struct NoPrefetch {
    __device__ __forceinline__ void operator()(int) {}
};

// Entry e of a value array (complex: both parts in one load; the arrays are the library's own
// allocations, so pairs are aligned).
template <typename T, bool CPLX>
struct MatVal {
    T r, i;
    __device__ __forceinline__ void load(const T* __restrict__ v, int64_t e) {
        if constexpr (!CPLX) { r = v[e]; i = T(0); }
        else if constexpr (sizeof(T) == 8) { const double2 t = reinterpret_cast<const double2*>(v)[e]; r = t.x; i = t.y; }
        else { const float2 t = reinterpret_cast<const float2*>(v)[e]; r = t.x; i = t.y; }
    }
    __device__ __forceinline__ void fma(T xr, T xi, T& ar, T& ai) const {
        if constexpr (CPLX) { ar += r * xr - i * xi; ai += r * xi + i * xr; }
        else { ar += r * xr; }
    }
};

// One SELL row: every column index first (w <= kSellMaxLen), then the gathers.  w and the slice's
// base are the wavefront's, STRIDE (the slice height) a constant where it is 64, so an entry is one
// load with an immediate offset and the width test a scalar branch.
template <typename T, bool CPLX, typename G>
__device__ __forceinline__ void sell_row(const int* __restrict__ col, const T* __restrict__ val, int lane, int stride,
                                         int w, const G& g, T& ar, T& ai) {
    int ci[kSellMaxLen];
#pragma unroll
    for (int j = 0; j < kSellMaxLen; j++)
        if (j < w) ci[j] = col[j * stride + lane];
#pragma unroll
    for (int j = 0; j < kSellMaxLen; j++)
        if (j < w) {
            MatVal<T, CPLX> v;
            v.load(val, j * stride + lane);
            T xr, xi;
            g(ci[j], xr, xi);
            v.fma(xr, xi, ar, ai);
        }
}

// A lane's share of a medium row, entries k0 + sub, k0 + sub + L, ...: U at a time, summed in order;
// past the end the lane's first entry is taken again with a zero value, so there is no branch.
template <typename T, bool CPLX, int L, typename G>
__device__ __forceinline__ void mid_row(const int* __restrict__ col, const T* __restrict__ val, int rem, const G& g, T& ar,
                                        T& ai) {
    constexpr int U = 4;
    for (; rem > 0; rem -= U * L, col += U * L, val += U * L * (CPLX ? 2 : 1)) {
        int c[U];
        MatVal<T, CPLX> v[U];
        T xr[U], xi[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int q = u * L < rem ? u * L : 0;
            c[u] = col[q];
            v[u].load(val, q);
        }
#pragma unroll
        for (int u = 0; u < U; u++) g(c[u], xr[u], xi[u]);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u * L >= rem) { v[u].r = T(0); v[u].i = T(0); xr[u] = T(0); xi[u] = T(0); }
            v[u].fma(xr[u], xi[u], ar, ai);
        }
    }
}

// Computes one row of A x for virtual block vb (uniform in the block), x given by a gather.
// Returns true in the thread that owns the result (row, ar, ai).  pre(row) is called in that thread
// as soon as the row is known, before any column is loaded, so that the caller's row-local
// operands (right-hand side, diagonal, vectors updated in place) are in flight together with the
// gathers instead of after them.
//
// Up to about 100,000 rows these kernels are bound by the instructions a wavefront issues, not by
// memory: an empty kernel takes 1.6 us, one with four dependent loads 2.2, and with 64-bit vector
// addresses, a runtime slice height and a divergent test per entry a smoothing step took 4.1 us
// on 4,900 rows of 5 and, with one column and gather at a time, 6.2 us on 9,683 rows of 12.
template <typename T, bool CPLX, typename G, typename P>
__device__ __forceinline__ bool spmv_row_gp(const SellDev<T>& A, const G& g, int vb, int& row, T& ar, T& ai, P& pre) {
    constexpr int W = CPLX ? 2 : 1;
    ar = 0;
    ai = 0;
    // the long rows' blocks come first: their wavefronts run the longest chains, so they start
    // with the launch and overlap the SELL rows instead of trailing them
    {
        const int nlb = A.nvb - A.nb_sell - A.nb_mid;
        vb = vb < nlb ? A.nb_sell + A.nb_mid + vb : vb - nlb;
    }
    if (vb < A.nb_sell) {
        const int r = vb * blockDim.x + threadIdx.x;
        // the slice is the wavefront's (C is a multiple of 64): its position is a scalar load
        const int r0 = __builtin_amdgcn_readfirstlane(r);
        if (r0 >= A.n_short) return false;
        const int s = A.C == 64 ? r0 >> 6 : r0 / A.C;
        const int64_t base = A.slice_ptr[s];
        const int w = A.slice_w[s];
        if (r >= A.n_short) return false;
        row = A.perm ? A.perm[r] : r;
        pre(row);
        const int* col = A.col + base;
        const T* val = A.val + base * W;
        if (A.C == 64) sell_row<T, CPLX>(col, val, r & 63, 64, w, g, ar, ai);
        else sell_row<T, CPLX>(col, val, r - s * A.C, A.C, w, g, ar, ai);
        return true;
    }
    if (vb < A.nb_sell + A.nb_mid) {  // medium rows: a group of mid_lanes lanes per row
        const int L = A.mid_lanes;
        const int t = (vb - A.nb_sell) * int(blockDim.x) + int(threadIdx.x);
        const int m = t >> (31 - __builtin_clz(unsigned(L))), sub = t & (L - 1);
        if (m < A.nmid) {
            const int64_t k = A.mid_ptr[m] + sub;
            const int rem = int(A.mid_ptr[m + 1] - k);
            row = A.mid_rows[m];
            if (sub == 0) pre(row);
            const int* col = A.mid_col + k;
            const T* val = A.mid_val + k * W;
            if (L == 4) mid_row<T, CPLX, 4>(col, val, rem, g, ar, ai);
            else if (L == 8) mid_row<T, CPLX, 8>(col, val, rem, g, ar, ai);
            else if (L == 16) mid_row<T, CPLX, 16>(col, val, rem, g, ar, ai);
            else if (L == 32) mid_row<T, CPLX, 32>(col, val, rem, g, ar, ai);
            else mid_row<T, CPLX, 64>(col, val, rem, g, ar, ai);
        }
        // reduce inside the group (every lane takes part; L divides 64)
        for (int off = L >> 1; off > 0; off >>= 1) {
            ar += __shfl_xor(ar, off, 64);
            if constexpr (CPLX) ai += __shfl_xor(ai, off, 64);
        }
        return m < A.nmid && sub == 0;
    }
    const int w = (vb - A.nb_sell - A.nb_mid) * int(blockDim.x >> 6) + int(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (w < A.nlong) {  // uniform inside the wavefront
        // a lane's entries k = lane, lane + 64, ...: U gathers in flight, summed in order (two
        // for complex values, whose registers would otherwise lower the occupancy of the whole
        // kernel, long rows or not)
        constexpr int U = CPLX ? 2 : 8;
        const int64_t kend = A.long_ptr[w + 1];
        int64_t k = A.long_ptr[w] + lane;
        row = A.long_rows[w];
        if (lane == 0) pre(row);
        auto add = [&](int64_t q, T xr, T xi) {
            MatVal<T, CPLX> v;
            v.load(A.long_val, q);
            v.fma(xr, xi, ar, ai);
        };
        for (; k + (U - 1) * 64 < kend; k += U * 64) {
            T xr[U], xi[U];
#pragma unroll
            for (int u = 0; u < U; u++) g(A.long_col[k + 64 * u], xr[u], xi[u]);
#pragma unroll
            for (int u = 0; u < U; u++) add(k + 64 * u, xr[u], xi[u]);
        }
        for (; k < kend; k += 64) {
            T xr, xi;
            g(A.long_col[k], xr, xi);
            add(k, xr, xi);
        }
        ar = wave_sum_t(ar);
        if constexpr (CPLX) ai = wave_sum_t(ai);
        return lane == 0;
    }
    return false;
}
template <typename T, bool CPLX, typename G>
__device__ __forceinline__ bool spmv_row_g(const SellDev<T>& A, const G& g, int vb, int& row, T& ar, T& ai) {
    NoPrefetch none;
    return spmv_row_gp<T, CPLX>(A, g, vb, row, ar, ai, none);
}


// The word the start's kernel stores its finding in, not known yet (the stream is idle or has read the last
// solve's: every solve ends with a readback).
static inline int* arm_start(mk_ctx* c) {
    __atomic_store_n(c->started(), -1, __ATOMIC_RELAXED);
    return c->started();
}
// Whether the start meets the tolerance, waited for while the first iterations run; false also when that
// takes longer than kStartWait.
static inline bool start_converged(mk_ctx* c) {
    constexpr auto kStartWait = std::chrono::microseconds(300);
    const auto t0 = std::chrono::steady_clock::now();
    int v;
    while ((v = __atomic_load_n(c->started(), __ATOMIC_RELAXED)) < 0)
        if (std::chrono::steady_clock::now() - t0 > kStartWait) return false;
    return v != 0;
}

static inline unsigned blocks_for(size_t len, int bs = 256) { return unsigned((len + bs - 1) / bs); }
// grid of the grid-stride reduction kernels: few enough blocks that the per-block arrival
// (partial store, device fence, ticket) stays a small part of the kernel
// Grid cap of the reducing kernels (grid-stride loops; partial sums per block): large enough
// to keep every CU's memory pipeline busy, small enough for a short partial-sum pass.
static inline unsigned red_grid() {
    static const unsigned g = [] {
        const char* s = std::getenv("METRIKO_RED_GRID");
        const long v = s ? std::atol(s) : 0;
        return v >= 64 && v <= 16384 ? unsigned(v) : 512u;
    }();
    return g;
}
static inline unsigned rgrid(size_t len) { return std::max(1u, std::min(blocks_for(len), red_grid())); }
// Grid cap of the fence-free two-launch reductions (partials_write / partials_sum).
static inline unsigned fin_grid() {
    static const unsigned g = [] {
        const char* s = std::getenv("METRIKO_FIN_GRID");
        const long v = s ? std::atol(s) : 0;
        return v >= 64 && v <= long(kMaxParts) ? unsigned(v) : 4096u;
    }();
    return g;
}
static inline unsigned fgrid(size_t len) { return std::max(1u, std::min(blocks_for(len), fin_grid())); }

hipEvent_t next_event(mk_ctx* c);
void timing_flush(mk_ctx* c);

// Counts an SpMV launch and, when timing is on, brackets it with events attributed to
// "<operator label>:<kernel>:<fp32|fp64>".
struct SpmvTimer {
    mk_ctx* c;
    // with timing on: start / end stamps for each of up to three launches of one timed
    // quantity (MK_TLAUNCH part 0, 1, 2); the durations are added (the intervals between the
    // launches are not counted)
    hipEvent_t ev[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    int parts = 1;
    mutable unsigned used = 0;
    SpmvTimer(mk_ctx* c_, double bytes, const mk_op* A = nullptr, const char* kernel = "spmv", bool fp32 = false,
              int nparts = 1)
        : c(c_), parts(nparts) {
        c->spmv_calls++;
        c->spmv_bytes += bytes;
        if (c->time_spmv) {
            if (c->ev_used + 2 * size_t(parts) > 4096) timing_flush(c);
            std::string key = std::string(A ? A->label : "op") + ":" + kernel + ":" + (fp32 ? "fp32" : "fp64");
            auto it = std::find_if(c->kstats.begin(), c->kstats.end(), [&](const auto& p) { return p.first == key; });
            if (it == c->kstats.end()) {
                mk_ctx::KStat s;
                s.bytes_per_call = bytes;
                s.rows = A ? A->n : 0;
                c->kstats.emplace_back(key, s);
                it = c->kstats.end() - 1;
            }
            it->second.bytes += bytes;
            for (int q = 0; q < parts; q++) {
                c->ev_key.push_back(q ? "+" + key : key);  // "+": time added to the call, no extra call
                ev[2 * q] = next_event(c);
                ev[2 * q + 1] = next_event(c);
            }
        }
    }
    ~SpmvTimer() {
        for (int q = 0; q < parts; q++)  // a part that was not launched: an empty interval
            if (ev[2 * q] && !(used & (1u << q))) {
                (void)hipEventRecord(ev[2 * q], c->stream);
                (void)hipEventRecord(ev[2 * q + 1], c->stream);
            }
    }
};

// Launches kernel K on STREAM.  With timing on, the launch carries the timer's start and end
// stamps of part PART through hipExtLaunchKernelGGL: they are taken at the kernel's own start
// and end, so the timed interval holds no event packet.
#define MK_TLAUNCH(tm, PART, K, G, B, SH, STREAM, ...)                                                  \
    do {                                                                                                \
        if ((tm).ev[0]) {                                                                               \
            (tm).used |= 1u << (PART);                                                                  \
            hipExtLaunchKernelGGL(K, G, B, SH, STREAM, (tm).ev[2 * (PART)], (tm).ev[2 * (PART) + 1], 0, \
                                  __VA_ARGS__);                                                         \
        } else {                                                                                        \
            hipLaunchKernelGGL(K, G, B, SH, STREAM, __VA_ARGS__);                                       \
        }                                                                                               \
    } while (0)

template <typename T>
static SellDev<T> sell_dev(const mk_op* A, const T* val, int block, unsigned* grid) {
    SellDev<T> d;
    d.n_short = A->n_short;
    d.C = A->C;
    d.nb_sell = int(blocks_for(size_t(A->n_short), block));
    d.nlong = A->nlong;
    d.slice_ptr = A->slice_ptr.p;
    d.slice_w = A->slice_w.p;
    d.col = A->col.p;
    d.val = val;
    d.perm = A->perm.p;
    d.long_rows = A->long_rows.p;
    d.long_ptr = A->long_ptr.p;
    d.long_col = A->long_col.p;
    d.nseg = A->nseg;
    d.seg_beg = A->seg_beg.p;
    d.seg_end = A->seg_end.p;
    d.lseg_ptr = A->lseg_ptr.p;
    d.seg_part = reinterpret_cast<T*>(A->seg_part.p);
    if constexpr (std::is_same<T, double>::value) d.long_val = A->long_val64.p;
    else d.long_val = A->long_val32.p;
    d.nmid = A->nmid;
    d.mid_lanes = A->mid_lanes;
    d.nb_mid = int(blocks_for(size_t(A->nmid) * size_t(A->mid_lanes), block));
    d.mid_rows = A->mid_rows.p;
    d.mid_ptr = A->mid_ptr.p;
    d.mid_col = A->mid_col.p;
    if constexpr (std::is_same<T, double>::value) d.mid_val = A->mid_val64.p;
    else d.mid_val = A->mid_val32.p;
    const unsigned nb_long = blocks_for(size_t(A->nlong), block / 64);
    *grid = std::max(1u, unsigned(d.nb_sell) + unsigned(d.nb_mid) + nb_long);
    d.nvb = int(*grid);
    return d;
}

}  // namespace mk
