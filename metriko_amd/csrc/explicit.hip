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
// more than kMaxRow entries are reported and the level is smoothed instead.
#include "mk_internal.h"
#include "sell.h"

namespace mk {

namespace {

constexpr int kHash = 1024;        // slots per row
constexpr int kMaxRow = kHash - 128;  // entries a row may have; a step adds at most 64 more

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

__device__ __forceinline__ unsigned hash_of(int c) { return (unsigned(c) * 2654435761u) >> 22; }  // 10 bits
static_assert(kHash == 1 << 10, "hash_of yields 10 bits");

// One row's table: keys, values (FILL) and the number of keys, of one wavefront.
template <bool CPLX, bool FILL>
struct RowTable {
    static constexpr int W = CPLX ? 2 : 1;
    int* key;
    double* val;
    int* count;
    // value (vr, vi) at column c; lanes of one call hold distinct columns
    __device__ __forceinline__ void add(int c, double vr, double vi) const {
        unsigned h = hash_of(c);
        int old;
        while ((old = atomicCAS(&key[h], -1, c)) != -1 && old != c) h = (h + 1) & (kHash - 1);
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
    // factor (fr, fi) times entries [b, e) of a CSR row; false when the row is too long
    __device__ __forceinline__ bool add_row(const CsrDev& M, int64_t b, int64_t e, double fr, double fi, int lane) const {
        for (int64_t k0 = b; k0 < e; k0 += 64) {
            // one wavefront: its LDS operations are in order, so the count is up to date and leaves
            // room for 64 more keys
            if (*static_cast<volatile int*>(count) > kMaxRow) return false;
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
template <bool CPLX, bool FILL>
__global__ void __launch_bounds__(256) k_spgemm(SpProduct S, int* __restrict__ cnt, int* __restrict__ overflow,
                                                const int64_t* __restrict__ optr, const int* __restrict__ ooff, int cshift,
                                                int* __restrict__ ocol, double* __restrict__ oval) {
    constexpr int W = CPLX ? 2 : 1;
    __shared__ int s_key[4][kHash];
    __shared__ double s_val[FILL ? 4 : 1][FILL ? kHash * W : 1];
    __shared__ int s_list[FILL ? 4 : 1][FILL ? kHash : 1];
    __shared__ int s_count[4];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int i = blockIdx.x * 4 + wid;
    if (i >= S.n) return;  // uniform inside the wavefront; nothing below synchronises the block
    const RowTable<CPLX, FILL> t{s_key[wid], s_val[FILL ? wid : 0], &s_count[wid]};
    for (int h = lane; h < kHash; h += 64) t.key[h] = -1;
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
        for (int h = lane; h < kHash; h += 64) {
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

// ptr[0 .. n] = exclusive prefix sums of a (+ b): one block, each thread a contiguous share
__global__ void __launch_bounds__(1024) k_scan(int n, const int* __restrict__ a, const int* __restrict__ b,
                                               int64_t* __restrict__ ptr) {
    __shared__ int64_t part[1024];
    const int t = threadIdx.x, per = (n + 1023) / 1024;
    const int i0 = min(n, t * per), i1 = min(n, i0 + per);
    int64_t s = 0;
    for (int i = i0; i < i1; i++) s += a[i] + (b ? b[i] : 0);
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int64_t v = t >= off ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    s = t ? part[t - 1] : 0;
    for (int i = i0; i < i1; i++) { ptr[i] = s; s += a[i] + (b ? b[i] : 0); }
    if (t == 1023) ptr[n] = part[1023];
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

// a CSR matrix on the device
struct DevCsr {
    DevBuf<int64_t> ptr;
    DevBuf<int> col;
    DevBuf<double> val;
    CsrDev view() const { return {ptr.p, col.p, val.p}; }
};

struct Builder {
    mk_ctx* c;
    bool cplx;
    DevBuf<int> overflow;
    Builder(mk_ctx* c_, bool cplx_) : c(c_), cplx(cplx_), overflow(1) {
        MK_HIP(hipMemsetAsync(overflow.p, 0, sizeof(int), c->stream));
    }
    DevCsr upload(const HostCsr& A) const {
        DevCsr d;
        const size_t nz = size_t(A.ptr[A.rows]);
        d.ptr.upload(A.ptr, size_t(A.rows) + 1, c->stream);
        d.col.upload(A.col, std::max<size_t>(nz, 1), c->stream);
        d.val.upload(A.val, std::max<size_t>(nz, 1) * (cplx ? 2 : 1), c->stream);
        return d;
    }
    void count(const SpProduct& S, DevBuf<int>& cnt) const {
        cnt.alloc(size_t(std::max(S.n, 1)));
        const dim3 g(unsigned((S.n + 3) / 4));
        if (cplx) hipLaunchKernelGGL((k_spgemm<true, false>), g, dim3(256), 0, c->stream, S, cnt.p, overflow.p, nullptr, nullptr, 0, nullptr, nullptr);
        else hipLaunchKernelGGL((k_spgemm<false, false>), g, dim3(256), 0, c->stream, S, cnt.p, overflow.p, nullptr, nullptr, 0, nullptr, nullptr);
        MK_HIP(hipGetLastError());
    }
    // row pointers from the counts; their total, or -1 when a row was too long
    int64_t scan(int n, const DevBuf<int>& a, const int* b, DevBuf<int64_t>& ptr) const {
        ptr.alloc(size_t(n) + 1);
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, c->stream, n, (const int*)a.p, b, ptr.p);
        int64_t* h = static_cast<int64_t*>(c->pin);
        MK_HIP(hipMemcpyAsync(h, ptr.p + n, sizeof(int64_t), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipMemcpyAsync(h + 1, overflow.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipStreamSynchronize(c->stream));
        return *reinterpret_cast<const int*>(h + 1) ? -1 : h[0];
    }
    void fill(const SpProduct& S, const int64_t* optr, const int* ooff, int cshift, int* ocol, double* oval) const {
        const dim3 g(unsigned((S.n + 3) / 4));
        if (cplx) hipLaunchKernelGGL((k_spgemm<true, true>), g, dim3(256), 0, c->stream, S, nullptr, nullptr, optr, ooff, cshift, ocol, oval);
        else hipLaunchKernelGGL((k_spgemm<false, true>), g, dim3(256), 0, c->stream, S, nullptr, nullptr, optr, ooff, cshift, ocol, oval);
        MK_HIP(hipGetLastError());
    }
    bool product(const SpProduct& S, DevCsr& out) const {
        DevBuf<int> cnt;
        count(S, cnt);
        const int64_t nz = scan(S.n, cnt, nullptr, out.ptr);
        if (nz < 0) return false;
        out.col.alloc(size_t(std::max<int64_t>(nz, 1)));
        out.val.alloc(size_t(std::max<int64_t>(nz, 1)) * (cplx ? 2 : 1));
        fill(S, out.ptr.p, nullptr, 0, out.col.p, out.val.p);
        return true;
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
    const Builder b(c, cplx);
    const int n = hA.rows, nc = hR.rows;
    const DevCsr A = b.upload(hA), P = b.upload(hP), R = b.upload(hR);
    DevBuf<double> D, vB(A.val.n), vG(A.val.n);
    D.upload(dinv, size_t(n), c->stream);
    const CsrDev a = A.view(), B{a.ptr, a.col, vB.p}, G{a.ptr, a.col, vG.p};  // B = D^-1 A, G = A D^-1
    const dim3 g(unsigned((n + 3) / 4));
    for (int rows = 0; rows < 2; rows++) {
        double* out = rows ? vB.p : vG.p;
        if (cplx) hipLaunchKernelGGL((k_scale<true>), g, dim3(256), 0, c->stream, n, a, (const double*)D.p, rows, out);
        else hipLaunchKernelGGL((k_scale<false>), g, dim3(256), 0, c->stream, n, a, (const double*)D.p, rows, out);
    }
    MK_HIP(hipGetLastError());
    DevCsr X, Wc, Q, U;
    // T = (2 alpha I - (2 beta + alpha^2) B + 2 alpha beta B^2 - beta^2 B^3) D^-1, by Horner;
    // V = (I - alpha B + beta B^2) P; M = [T | V]
    if (!b.product({n, -beta * beta, B, B, 2.0 * alpha * beta, B, 0.0, {}, -(2.0 * beta + alpha * alpha)}, Q)) return false;
    if (!b.product({n, 1.0, B, P.view()}, U)) return false;
    const SpProduct T{n, 1.0, B, Q.view(), 0.0, {}, 0.0, {}, 2.0 * alpha, D.p};
    const SpProduct V{n, beta, B, U.view(), -alpha, U.view(), 1.0, P.view()};
    DevBuf<int> cT, cV;
    b.count(T, cT);
    b.count(V, cV);
    DevCsr Mc;
    const int64_t nz = b.scan(n, cT, cV.p, Mc.ptr);
    if (nz < 0 || double(nz) * (cplx ? 12.0 : 8.0) > max_bytes) return false;
    // W = R (I - alpha G + beta G^2)
    if (!b.product({nc, 1.0, R.view(), G}, X)) return false;
    if (!b.product({nc, beta, X.view(), G, -alpha, X.view(), 1.0, R.view()}, Wc)) return false;
    Mc.col.alloc(size_t(std::max<int64_t>(nz, 1)));
    Mc.val.alloc(size_t(std::max<int64_t>(nz, 1)) * (cplx ? 2 : 1));
    b.fill(T, Mc.ptr.p, nullptr, 0, Mc.col.p, Mc.val.p);
    b.fill(V, Mc.ptr.p, cT.p, n, Mc.col.p, Mc.val.p);
    const int64_t wz = int64_t(Wc.col.n);
    *W = b.op(nc, n, wz, std::move(Wc.ptr), std::move(Wc.col), std::move(Wc.val), block);
    *M = b.op(n, n + nc, nz, std::move(Mc.ptr), std::move(Mc.col), std::move(Mc.val), block);
    MK_HIP(hipStreamSynchronize(c->stream));  // the temporaries are freed on return
    return true;
}

}  // namespace mk
