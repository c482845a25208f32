// A multigrid level as two explicit sparse products, formed on the device.
//
// Chebyshev(2) smoothing is x + q (b - A x) with q = alpha D^-1 - beta D^-1 A D^-1, so one level of
// the V-cycle (smooth from zero, restrict the residual, correct, smooth) computes
//   b_c = R (I - A q) b = W b,      x = (2 q - q A q) b + (I - q A) P x_c = M [b; x_c]:
// the same preconditioner in two kernels instead of six.  The rows are six to eight times as long
// (a 40,820-face field: 4.0 -> 26.6 entries, its second level 11.7 -> 92.9), but a small level pays per
// kernel, 3 to 6 us each whatever its size, and not per byte.
//
// Where the line lies (a solve with such levels smoothed -> explicit): 4,900 rows of 5 0.82 -> 0.52 ms;
// 62,307 complex rows of 5 and their 10,369 in FP64 1.36 -> 0.89 ms; a field of 40,820 faces 42 -> 23 ms;
// 72,974 rows of 9 (33 MB) and less below 655,743 5.7 -> 4.8 ms; but 220,152 complex rows of 10.7 (240 MB)
// below a 1,310,720-face field 437 -> 538 ms, so M is kept to what stays in the Infinity Cache beside
// the solve's vectors.  (20,567 x 37 columns use the smoother either way.)
//
// The products are row-wise SpGEMMs, one wavefront per row with a hash table of the row in LDS: the
// entries of the left row are taken in order, the lanes spread over the right row (whose columns are
// distinct), so every sum has a fixed order; the finished row is written in column order.  Rows of
// more than kMaxRow entries are reported and the level is smoothed instead.  Counting uses a table of
// kHash slots, filling one of kSmall where every row fits: a quarter of the clearing, collecting and LDS
// (16 KB a block instead of 64, so ten blocks per compute unit instead of two): 62,307 complex rows of
// 5, four products of up to 33 entries a row, 500 -> 110 us each.
//
// A first solve pays for all of this, so the temporaries are carved out of scratch that the context keeps
// (allocating and freeing them took 3 of the 8.6 ms that 102,845 rows of 9 cost before): a first solve
// of that operator 26.0 -> 20.9 ms, 21.1 with the level smoothed.
#include "mk_internal.h"
#include "sell.h"

namespace mk {

namespace {

constexpr int kHash = 1024;           // slots per row
constexpr int kMaxRow = kHash - 128;  // entries a row may have; a step adds at most 64 more
constexpr int kSmall = 256;           // slots per row where no row has more than kSmallRow entries
constexpr int kSmallRow = 192;

struct CsrDev {
    const int64_t* ptr = nullptr;  // null: absent
    const int* col = nullptr;
    const double* val = nullptr;
};

// C = (s A B + z1 Z1 + z2 Z2 + d I) diag(cs) of n rows; Z1, Z2 and cs may be absent
struct SpProduct {
    int n = 0;
    double s = 1.0;
    CsrDev A, B;
    double z1 = 0.0;
    CsrDev Z1;
    double z2 = 0.0;
    CsrDev Z2;
    double d = 0.0;
    const double* cs = nullptr;
};

// the slot of a column in a table of H (a power of two) slots
template <int H>
__device__ __forceinline__ unsigned hash_of(int c) {
    return (unsigned(c) * 2654435761u) >> (32 - __builtin_ctz(H));
}

// One row's table of H slots: keys, values (FILL) and the number of keys, of one wavefront.
template <bool CPLX, bool FILL, int H>
struct RowTable {
    static constexpr int W = CPLX ? 2 : 1;
    int* key;
    double* val;
    int* count;
    // value (vr, vi) at column c; lanes of one call hold distinct columns
    __device__ __forceinline__ void add(int c, double vr, double vi) const {
        unsigned h = hash_of<H>(c);
        int old;
        while ((old = atomicCAS(&key[h], -1, c)) != -1 && old != c) h = (h + 1) & (H - 1);
        if (old == -1) atomicAdd(count, 1);
        if constexpr (FILL) {
            if (old == -1) {
                val[W * h] = vr;
                if constexpr (CPLX) val[W * h + 1] = vi;
            } else {
                val[W * h] += vr;
                if constexpr (CPLX) val[W * h + 1] += vi;
            }
        }
    }
    // factor (fr, fi) times entries [b, e) of a CSR row; false when the row is too long (counting only: a
    // row that is filled fits)
    __device__ __forceinline__ bool add_row(const CsrDev& M, int64_t b, int64_t e, double fr, double fi, int lane) const {
        for (int64_t k0 = b; k0 < e; k0 += 64) {
            // one wavefront: its LDS operations are in order, so the count is up to date and leaves
            // room for 64 more keys
            if (!FILL && *static_cast<volatile int*>(count) > kMaxRow) return false;
            const int64_t k = k0 + lane;
            if (k < e) {
                double vr = 0.0, vi = 0.0;
                if constexpr (FILL) {
                    vr = M.val[W * k];
                    if constexpr (CPLX) {
                        vi = M.val[W * k + 1];
                        const double t = fr * vr - fi * vi;
                        vi = fr * vi + fi * vr;
                        vr = t;
                    } else {
                        vr *= fr;
                    }
                }
                add(M.col[k], vr, vi);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        return true;
    }
};

// FILL = false: cnt[i] = entries of row i (overflow set when it has too many).  FILL = true: row i
// in column order at optr[i] + (ooff ? ooff[i] : 0), columns shifted by cshift.
template <bool CPLX, bool FILL, int H>
__global__ void __launch_bounds__(256) k_spgemm(SpProduct S, int* __restrict__ cnt, int* __restrict__ overflow,
                                                const int64_t* __restrict__ optr, const int* __restrict__ ooff, int cshift,
                                                int* __restrict__ ocol, double* __restrict__ oval) {
    constexpr int W = CPLX ? 2 : 1;
    __shared__ int s_key[4][H];
    __shared__ double s_val[FILL ? 4 : 1][FILL ? H * W : 1];
    __shared__ int s_list[FILL ? 4 : 1][FILL ? H : 1];
    __shared__ int s_count[4];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int i = blockIdx.x * 4 + wid;
    if (i >= S.n) return;  // uniform inside the wavefront; nothing below synchronises the block
    const RowTable<CPLX, FILL, H> t{s_key[wid], s_val[FILL ? wid : 0], &s_count[wid]};
    for (int h = lane; h < H; h += 64) t.key[h] = -1;
    if (lane == 0) s_count[wid] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    bool ok = true;
    for (int64_t k = S.A.ptr[i]; k < S.A.ptr[i + 1] && ok; k++) {
        const int j = S.A.col[k];
        double ar = 0.0, ai = 0.0;
        if constexpr (FILL) {
            ar = S.s * S.A.val[W * k];
            if constexpr (CPLX) ai = S.s * S.A.val[W * k + 1];
        }
        ok = t.add_row(S.B, S.B.ptr[j], S.B.ptr[j + 1], ar, ai, lane);
    }
    if (S.Z1.ptr) ok = ok && t.add_row(S.Z1, S.Z1.ptr[i], S.Z1.ptr[i + 1], S.z1, 0.0, lane);
    if (S.Z2.ptr) ok = ok && t.add_row(S.Z2, S.Z2.ptr[i], S.Z2.ptr[i + 1], S.z2, 0.0, lane);
    if (S.d != 0.0 && lane == 0) t.add(i, S.d, 0.0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int m = *static_cast<volatile int*>(&s_count[wid]);
    if constexpr (!FILL) {
        if (lane == 0) {
            cnt[i] = m;
            if (!ok) *overflow = 1;
        }
    } else {
        // occupied slots, then every key's rank among them
        int* list = s_list[wid];
        int base = 0;
        for (int h = lane; h < H; h += 64) {
            const bool used = t.key[h] >= 0;
            const unsigned long long b = __ballot(used);
            if (used) list[base + __popcll(b & ((1ull << lane) - 1))] = h;
            base += __popcll(b);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int64_t o = optr[i] + (ooff ? ooff[i] : 0);
        for (int e = lane; e < m; e += 64) {
            const int h = list[e], c = t.key[h];
            int rank = 0;
            for (int q = 0; q < m; q++) rank += t.key[list[q]] < c ? 1 : 0;
            const double s = S.cs ? S.cs[c] : 1.0;
            ocol[o + rank] = c + cshift;
            for (int w = 0; w < W; w++) oval[W * (o + rank) + w] = s * t.val[W * h + w];
        }
    }
}

// ptr[0 .. n] = exclusive prefix sums of a (+ b), maxima[0], maxima[1] = the largest of a and of b: one block,
// a tile of 4,096 rows at a time, four neighbouring rows a thread.  (With a contiguous share of the
// whole per thread 62,307 rows took 209 us, this 55.)
__global__ void __launch_bounds__(1024) k_scan(int n, const int* __restrict__ a, const int* __restrict__ b,
                                               int64_t* __restrict__ ptr, int* __restrict__ maxima) {
    __shared__ int wsum[2][16];
    __shared__ int smax[2][16];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    int64_t base = 0;
    int ma = 0, mb = 0;
    int buf = 0;
    for (int i0 = 0; i0 < n; i0 += 4096, buf ^= 1) {
        int v[4], s = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = i0 + 4 * t + q;
            const int x = i < n ? a[i] : 0, y = b && i < n ? b[i] : 0;
            ma = max(ma, x);
            mb = max(mb, y);
            v[q] = x + y;
            s += v[q];
        }
        int inc = s;  // inclusive sums over the wavefront (a tile holds fewer than 2^31 entries)
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(inc, off, 64);
            if (lane >= off) inc += u;
        }
        if (lane == 63) wsum[buf][wid] = inc;
        __syncthreads();
        int before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < 16; w++) {
            if (w < wid) before += wsum[buf][w];
            all += wsum[buf][w];
        }
        int64_t o = base + before + inc - s;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int i = i0 + 4 * t + q;
            if (i < n) ptr[i] = o;
            o += v[q];
        }
        base += all;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        ma = max(ma, __shfl_xor(ma, off, 64));
        mb = max(mb, __shfl_xor(mb, off, 64));
    }
    if (lane == 0) { smax[0][wid] = ma; smax[1][wid] = mb; }
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < 16; w++) { ma = max(ma, smax[0][w]); mb = max(mb, smax[1][w]); }
        ptr[n] = base;
        maxima[0] = ma;
        maxima[1] = mb;
    }
}

// y = diag(d) x (rows != 0) or x diag(d), on the values of a CSR matrix: one wavefront per row
template <bool CPLX>
__global__ void __launch_bounds__(256) k_scale(int n, CsrDev A, const double* __restrict__ d, int rows,
                                               double* __restrict__ out) {
    constexpr int W = CPLX ? 2 : 1;
    const int i = blockIdx.x * 4 + int(threadIdx.x >> 6);
    if (i >= n) return;
    for (int64_t k = A.ptr[i] + (threadIdx.x & 63); k < A.ptr[i + 1]; k += 64) {
        const double f = rows ? d[i] : d[A.col[k]];
        for (int w = 0; w < W; w++) out[W * k + w] = f * A.val[W * k + w];
    }
}
__global__ void k_iota(int n, int* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = i;
}
__global__ void k_round32(size_t n, const double* __restrict__ x, float* __restrict__ y) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) y[i] = float(x[i]);
}
inline unsigned nb(size_t n) { return unsigned((n + 255) / 256); }

// Temporaries of one set-up, carved out of the context's scratch chunks in order.  The context keeps up to
// kKeep of them for the next set-up (its stream runs the two one after the other) until it ends.
struct Scratch {
    static constexpr size_t kChunk = size_t(32) << 20, kKeep = size_t(256) << 20;
    mk_ctx* c;
    size_t k = 0, off = 0;
    explicit Scratch(mk_ctx* c_) : c(c_) {}
    Scratch(const Scratch&) = delete;
    ~Scratch() {
        size_t held = 0;
        for (size_t q = 0; q < c->scratch.size();) {
            if (held + c->scratch[q].n <= kKeep) held += c->scratch[q++].n;
            else c->scratch.erase(c->scratch.begin() + std::ptrdiff_t(q));
        }
    }
    template <typename T>
    T* get(size_t count) {
        const size_t bytes = (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
        while (k < c->scratch.size() && off + bytes > c->scratch[k].n) { k++; off = 0; }
        if (k == c->scratch.size()) c->scratch.emplace_back(std::max(bytes, kChunk));
        T* p = reinterpret_cast<T*>(c->scratch[k].p + off);
        off += bytes;
        return p;
    }
};

// a CSR matrix on the device that the caller keeps
struct DevCsr {
    DevBuf<int64_t> ptr;
    DevBuf<int> col;
    DevBuf<double> val;
};
// entries of a product and of its longest row; nz < 0: a row was too long
struct Size { int64_t nz; int longest, longest_b; };

struct Builder {
    mk_ctx* c;
    bool cplx;
    Scratch& tmp;
    int* overflow;
    Builder(mk_ctx* c_, bool cplx_, Scratch& t) : c(c_), cplx(cplx_), tmp(t), overflow(t.get<int>(1)) {
        MK_HIP(hipMemsetAsync(overflow, 0, sizeof(int), c->stream));
    }
    template <typename T>
    const T* upload(const T* h, size_t n) const {
        T* d = tmp.get<T>(n);
        if (n) MK_HIP(hipMemcpyAsync(d, h, n * sizeof(T), hipMemcpyHostToDevice, c->stream));
        return d;
    }
    CsrDev upload(const HostCsr& A) const {
        const size_t nz = size_t(A.ptr[A.rows]);
        return {upload(A.ptr, size_t(A.rows) + 1), upload(A.col, nz), upload(A.val, nz * (cplx ? 2 : 1))};
    }
    int* count(const SpProduct& S) const {
        int* cnt = tmp.get<int>(size_t(S.n));
        const dim3 g(unsigned((S.n + 3) / 4));
#define MK_COUNT(CP)                                                                                                \
    hipLaunchKernelGGL((k_spgemm<CP, false, kHash>), g, dim3(256), 0, c->stream, S, cnt, overflow, nullptr, nullptr, \
                       0, nullptr, nullptr)
        if (cplx) MK_COUNT(true);
        else MK_COUNT(false);
#undef MK_COUNT
        MK_HIP(hipGetLastError());
        return cnt;
    }
    // row pointers from the counts a (+ b)
    Size scan(int n, const int* a, const int* b, int64_t* ptr) const {
        int* found = tmp.get<int>(2);
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, c->stream, n, a, b, ptr, found);
        int64_t* h = static_cast<int64_t*>(c->pin);
        int* hi = reinterpret_cast<int*>(h + 1);
        MK_HIP(hipMemcpyAsync(h, ptr + n, sizeof(int64_t), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipMemcpyAsync(hi, found, 2 * sizeof(int), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipMemcpyAsync(hi + 2, overflow, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipStreamSynchronize(c->stream));
        return {hi[2] ? -1 : *h, hi[0], hi[1]};
    }
    // longest: the longest row's entries
    void fill(const SpProduct& S, int longest, const int64_t* optr, const int* ooff, int cshift, int* ocol,
              double* oval) const {
        const dim3 g(unsigned((S.n + 3) / 4));
#define MK_FILL(CP, H)                                                                                            \
    hipLaunchKernelGGL((k_spgemm<CP, true, H>), g, dim3(256), 0, c->stream, S, nullptr, nullptr, optr, ooff, cshift, \
                       ocol, oval)
        const bool small = longest <= kSmallRow;
        if (cplx) { if (small) MK_FILL(true, kSmall); else MK_FILL(true, kHash); }
        else { if (small) MK_FILL(false, kSmall); else MK_FILL(false, kHash); }
#undef MK_FILL
        MK_HIP(hipGetLastError());
    }
    // false: a row was too long
    bool product(const SpProduct& S, CsrDev& out) const {
        const int* cnt = count(S);
        int64_t* ptr = tmp.get<int64_t>(size_t(S.n) + 1);
        const Size z = scan(S.n, cnt, nullptr, ptr);
        if (z.nz < 0) return false;
        int* col = tmp.get<int>(size_t(z.nz));
        double* val = tmp.get<double>(size_t(z.nz) * (cplx ? 2 : 1));
        fill(S, z.longest, ptr, nullptr, 0, col, val);
        out = {ptr, col, val};
        return true;
    }
    void alloc(DevCsr& out, int64_t nz) const {
        out.col.alloc(size_t(std::max<int64_t>(nz, 1)));
        out.val.alloc(size_t(std::max<int64_t>(nz, 1)) * (cplx ? 2 : 1));
    }
    // an operator of medium rows only, taking over its CSR arrays
    mk_op* op(int rows, int cols, int64_t nz, DevBuf<int64_t>&& ptr, DevBuf<int>&& col, DevBuf<double>&& val, int block) const {
        const int vw = cplx ? 2 : 1;
        auto* o = new mk_op();
        try {
            o->ctx = c;
            o->n = rows;
            o->m = cols;
            o->cplx = cplx;
            o->nnz = nz;
            o->block = block;
            o->nmid = rows;
            // about four entries per lane, as build_sell takes for its medium rows
            const double avg = rows ? double(nz) / rows : 0.0;
            o->mid_lanes = 4;
            while (o->mid_lanes < 64 && o->mid_lanes * 4 < avg) o->mid_lanes *= 2;
            o->mid_ptr = std::move(ptr);
            o->mid_col = std::move(col);
            o->mid_val64 = std::move(val);
            o->mid_rows.alloc(size_t(rows));
            o->mid_val32.alloc(size_t(std::max<int64_t>(nz, 1)) * vw);
            hipLaunchKernelGGL(k_iota, dim3(nb(size_t(rows))), dim3(256), 0, c->stream, rows, o->mid_rows.p);
            hipLaunchKernelGGL(k_round32, dim3(nb(size_t(nz) * vw)), dim3(256), 0, c->stream, size_t(nz) * vw,
                               (const double*)o->mid_val64.p, o->mid_val32.p);
            MK_HIP(hipGetLastError());
            o->bytes64 = double(nz) * (8.0 * vw + 4.0) + rows * 12.0 + double(rows + cols) * 8.0 * vw;
            o->bytes32 = double(nz) * (4.0 * vw + 4.0) + rows * 12.0 + double(rows + cols) * 4.0 * vw;
        } catch (...) {
            delete o;
            throw;
        }
        return o;
    }
};

}  // namespace

bool explicit_level(mk_ctx* c, bool cplx, const HostCsr& hA, const HostCsr& hP, const HostCsr& hR, const double* dinv,
                    double alpha, double beta, double max_bytes, int block, mk_op** W, mk_op** M) {
    Scratch tmp(c);
    const Builder b(c, cplx, tmp);
    const int n = hA.rows, nc = hR.rows;
    const CsrDev a = b.upload(hA), P = b.upload(hP), R = b.upload(hR);
    const double* D = b.upload(dinv, size_t(n));
    // B = D^-1 A, G = A D^-1
    const size_t len = size_t(hA.ptr[n]) * (cplx ? 2 : 1);
    double *vB = tmp.get<double>(len), *vG = tmp.get<double>(len);
    const CsrDev B{a.ptr, a.col, vB}, G{a.ptr, a.col, vG};
    const dim3 g(unsigned((n + 3) / 4));
    for (int rows = 0; rows < 2; rows++) {
        double* out = rows ? vB : vG;
        if (cplx) hipLaunchKernelGGL((k_scale<true>), g, dim3(256), 0, c->stream, n, a, D, rows, out);
        else hipLaunchKernelGGL((k_scale<false>), g, dim3(256), 0, c->stream, n, a, D, rows, out);
    }
    MK_HIP(hipGetLastError());
    CsrDev X, Q, U;
    // T = (2 alpha I - (2 beta + alpha^2) B + 2 alpha beta B^2 - beta^2 B^3) D^-1, by Horner;
    // V = (I - alpha B + beta B^2) P; M = [T | V]
    if (!b.product({n, -beta * beta, B, B, 2.0 * alpha * beta, B, 0.0, {}, -(2.0 * beta + alpha * alpha)}, Q)) return false;
    if (!b.product({n, 1.0, B, P}, U)) return false;
    const SpProduct T{n, 1.0, B, Q, 0.0, {}, 0.0, {}, 2.0 * alpha, D};
    const SpProduct V{n, beta, B, U, -alpha, U, 1.0, P};
    const int *cT = b.count(T), *cV = b.count(V);
    DevCsr Wc, Mc;
    Mc.ptr.alloc(size_t(n) + 1);
    const Size m = b.scan(n, cT, cV, Mc.ptr.p);
    if (m.nz < 0 || double(m.nz) * (cplx ? 12.0 : 8.0) > max_bytes) return false;
    // W = R (I - alpha G + beta G^2)
    if (!b.product({nc, 1.0, R, G}, X)) return false;
    const SpProduct Wp{nc, beta, X, G, -alpha, X, 1.0, R};
    const int* cW = b.count(Wp);
    Wc.ptr.alloc(size_t(nc) + 1);
    const Size w = b.scan(nc, cW, nullptr, Wc.ptr.p);
    if (w.nz < 0) return false;
    b.alloc(Wc, w.nz);
    b.alloc(Mc, m.nz);
    b.fill(Wp, w.longest, Wc.ptr.p, nullptr, 0, Wc.col.p, Wc.val.p);
    b.fill(T, m.longest, Mc.ptr.p, nullptr, 0, Mc.col.p, Mc.val.p);
    b.fill(V, m.longest_b, Mc.ptr.p, cT, n, Mc.col.p, Mc.val.p);
    *W = b.op(nc, n, w.nz, std::move(Wc.ptr), std::move(Wc.col), std::move(Wc.val), block);
    *M = b.op(n, n + nc, m.nz, std::move(Mc.ptr), std::move(Mc.col), std::move(Mc.val), block);
    MK_HIP(hipStreamSynchronize(c->stream));  // the host arrays and the scratch may go
    return true;
}

}  // namespace mk
