// Sparse kernels and the PCG / refinement solvers of the metriko HIP library (gfx950).
//
// Layout: SELL-C-sigma (slice height C = 64 = one wavefront by default): entries of
// slice s are stored column-major (val[slice_ptr[s] + j*C + lane]) so every load of
// a wavefront is one contiguous, coalesced 64-lane access.  Rows may be sorted by
// length inside windows of sigma rows (perm maps a stored row to the original row).
//
// Reductions are deterministic: each block reduces with DPP row shifts and broadcasts inside its
// wavefronts and LDS between them and writes one partial; the kernel that needs the total, or a one-block
// kernel in between, sums the partials in a fixed order.  Reruns are therefore bit-identical.
#include <algorithm>
#include <chrono>
#include <memory>
#include <cmath>
#include <cstring>
#include <numeric>
#include "mk_internal.h"

#include "sell.h"

namespace mk {

hipEvent_t next_event(mk_ctx* c) {
    if (c->ev_used == c->ev_pool.size()) {
        hipEvent_t e;
        MK_HIP(hipEventCreate(&e));
        c->ev_pool.push_back(e);
    }
    return c->ev_pool[c->ev_used++];
}

void timing_flush(mk_ctx* c) {
    if (!c->time_spmv || c->ev_used == 0) { c->ev_used = 0; return; }
    MK_HIP(hipStreamSynchronize(c->stream));
    for (size_t i = 0; i + 1 < c->ev_used; i += 2) {
        float ms = 0.f;
        MK_HIP(hipEventElapsedTime(&ms, c->ev_pool[i], c->ev_pool[i + 1]));
        c->spmv_ms += ms;
        const std::string& k = c->ev_key[i / 2];
        const bool cont = !k.empty() && k[0] == '+';  // second launch of the previous call
        const std::string key = cont ? k.substr(1) : k;
        auto it = std::find_if(c->kstats.begin(), c->kstats.end(), [&](const auto& p) { return p.first == key; });
        if (it != c->kstats.end()) { if (!cont) it->second.calls++; it->second.ms += ms; }
    }
    c->ev_used = 0;
    c->ev_key.clear();
}


// ---- second launch of the two-launch reductions ---------------------------------------------
// k_finish: one block sums the partials of the nparts blocks of the previous kernel (fixed order).
__global__ void __launch_bounds__(1024) k_finish(const double* __restrict__ partials, int nparts, double* out,
                                                 const int* skip) {
    if (skip && *skip) return;
    double tot[1];
    partials_sum<1>(partials, nparts, tot);
    if (threadIdx.x == 0) out[0] = tot[0];
}
static inline void finish(mk_ctx* c, unsigned nparts, double* out, const int* skip = nullptr,
                          const double* partials = nullptr) {
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(1024), 0, c->stream, partials ? partials : (const double*)c->partials.p,
                       int(nparts), out, skip);
}

// One vector's element `row` (complex: two entries), loaded by spmv_row_gp's early hook.
template <typename T, bool CPLX>
struct RowElem {
    static constexpr int W = CPLX ? 2 : 1;
    const T* __restrict__ src;   // nullptr: nothing to load
    T v[W];
    __device__ __forceinline__ void operator()(int row) {
        if (!src) return;
#pragma unroll
        for (int q = 0; q < W; q++) v[q] = src[W * row + q];
    }
};

template <typename T, bool CPLX, int MODE>
__global__ void __launch_bounds__(256) sell_spmv(SellDev<T> A, const T* __restrict__ x, T* __restrict__ y,
                                               const T* __restrict__ b, double* partials, const int* skip) {
    if (skip && *skip) return;
    double contrib = 0.0;
    // reducing modes run a capped grid that strides over the virtual blocks
    for (int vb = blockIdx.x; vb < A.nvb; vb += gridDim.x) {
        int row = 0;
        T ar, ai;
        // the row's own element of b (modes 2, 3), y (4) or x (1), fetched early
        RowElem<T, CPLX> re{MODE == 2 || MODE == 3 ? b : MODE == 4 ? y : MODE == 1 ? x : nullptr};
        if (!spmv_row_gp<T, CPLX>(A, PlainGather<T, CPLX>{x}, vb, row, ar, ai, re)) continue;
        if constexpr (CPLX) {
            if constexpr (MODE == 2 || MODE == 3) { ar = re.v[0] - ar; ai = re.v[1] - ai; }
            if constexpr (MODE == 4) { ar += re.v[0]; ai += re.v[1]; }
            if (MODE != 2 || y) { y[2 * row] = ar; y[2 * row + 1] = ai; }  // residual norm alone: no y
            if constexpr (MODE == 1) contrib += double(re.v[0]) * double(ar) + double(re.v[1]) * double(ai);
            if constexpr (MODE == 2) contrib += double(ar) * double(ar) + double(ai) * double(ai);
        } else {
            T a = ar;
            if constexpr (MODE == 2 || MODE == 3) a = re.v[0] - a;
            if constexpr (MODE == 4) a += re.v[0];
            if (MODE != 2 || y) y[row] = a;
            if constexpr (MODE == 1) contrib += double(re.v[0]) * double(a);
            if constexpr (MODE == 2) contrib += double(a) * double(a);
        }
    }
    if constexpr (MODE == 1 || MODE == 2) {
        double v[1] = {contrib};
        partials_write<1>(v, partials);
    }
}

// ---------------------------------------------------------------------------------------
// CG kernels.  Vectors are real arrays of length len = n (real) or 2n (complex);
// element e of a complex vector occupies entries 2e, 2e+1; the Jacobi scaling dinv
// is per element (real).
template <typename T, bool CPLX>
__global__ void __launch_bounds__(256) cg_init(int n, const T* __restrict__ r, const T* __restrict__ b,
                                             const T* __restrict__ dinv, T* __restrict__ z, T* __restrict__ p,
                                             double* partials) {
    double rz = 0.0, rr = 0.0, bb = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const T d = dinv ? dinv[i] : T(1);
        if constexpr (CPLX) {
            const T r0 = r[2 * i], r1 = r[2 * i + 1];
            const T z0 = d * r0, z1 = d * r1;
            z[2 * i] = z0; z[2 * i + 1] = z1; p[2 * i] = z0; p[2 * i + 1] = z1;
            rz += double(r0) * z0 + double(r1) * z1;
            rr += double(r0) * r0 + double(r1) * r1;
            bb += double(b[2 * i]) * b[2 * i] + double(b[2 * i + 1]) * b[2 * i + 1];
        } else {
            const T r0 = r[i], z0 = d * r0;
            z[i] = z0; p[i] = z0;
            rz += double(r0) * z0;
            rr += double(r0) * r0;
            bb += double(b[i]) * b[i];
        }
    }
    double v[3] = {rz, rr, bb};
    partials_write<3>(v, partials);
}

// One iteration is cg_step1 (p = z + beta p ; q = A p ; p^H q) and cg_step2 (x += alpha p ;
// r -= alpha q ; with Jacobi z = dinv r and rz), plus, with an external preconditioner, its
// application and cg_beta (rz).  The scalars between them: rz in row 0 of the partials, rr in row 1,
// p^H q in row 2.  Up to kFoldParts blocks every block of the kernel that needs a scalar adds the
// previous kernel's partials itself, in the same order (the same value in every block, one block
// stores what the host reads); above that, one-block kernels add them in between.  A one-block
// kernel costs 2.3 to 3 us, a fold of 200 partials 0.6: with folds and the update of p inside the
// product (from the old p of the gathered rows; p alternates between two buffers) a Jacobi
// iteration on 50,953 rows went from five launches to two (703 iterations 14 to 8.4 ms, 20 to 12 us
// each).  The line: every block reads all partials, so the fold grows with the square of the grid;
// with it at 4096 a field on 655,362 vertices took 501 ms (455 at 2048) and 655,743 unknowns 5.15 ms
// (4.8); at 1024 no size measured was faster than at 2048.
static constexpr unsigned kFoldParts = 2048;
static constexpr int kRowRz = 0, kRowRr = 1, kRowPq = 2;

// The gathered p = z + beta p_old, never stored before it is used
template <typename T, bool CPLX>
struct DirectionGather {
    const T* __restrict__ z;
    const T* __restrict__ p;
    T beta;
    __device__ __forceinline__ void operator()(int c, T& xr, T& xi) const {
        if constexpr (CPLX) { xr = z[2 * c] + beta * p[2 * c]; xi = z[2 * c + 1] + beta * p[2 * c + 1]; }
        else { xr = z[c] + beta * p[c]; xi = T(0); }
    }
};
template <typename T, bool CPLX>
struct DirectionOperands {
    static constexpr int W = CPLX ? 2 : 1;
    const T* __restrict__ z;
    const T* __restrict__ p;
    T zv[W], pv[W];
    __device__ __forceinline__ void operator()(int row) {
#pragma unroll
        for (int q = 0; q < W; q++) { zv[q] = z[W * row + q]; pv[q] = p[W * row + q]; }
    }
};

// nin: partials of rz (Jacobi: and rr) to fold (0: the state holds beta).
//
// No block of a launch reads a word that another block of it writes (a block that starts late would
// see either value, each of its wavefronts for itself).  The iteration's rz goes to st->rz_new, and
// cg_step2 moves it to st->rz; the end of the solve, found by a fold, is in the same way handed on
// in st->stop, which cg_step2 tests and moves to st->done, the word all other kernels test.
template <typename T, bool CPLX, bool JAC>
__global__ void __launch_bounds__(256) cg_step1(SellDev<T> A, const T* __restrict__ z, const T* __restrict__ p,
                                              T* __restrict__ pn, T* __restrict__ q, CgState* st, double* partials, int nin) {
    constexpr int W = CPLX ? 2 : 1;
    const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
    if (st->done) {
        if (writer) st->stop = 1;
        return;
    }
    T beta;
    if (nin) {
        double tot[JAC ? 2 : 1];
        partials_sum<JAC ? 2 : 1>(partials, nin, tot);
        const double rz = tot[0];
        bool stop = false;
        if constexpr (JAC) {
            const double rr = tot[1];
            const bool nan = !(rr == rr) || !(rz == rz);
            stop = nan || rr <= st->tol2 * st->bb;
            if (writer) {
                st->rr = rr;
                st->it += 1;
                if (nan) st->status = MK_ERR_NAN;
                if (stop) st->stop = 1;
            }
        } else {
            stop = !(rz > 0.0);
            if (writer && stop) { st->status = (rz == rz) ? MK_ERR_NOT_SPD : MK_ERR_NAN; st->stop = 1; }
        }
        if (stop) return;
        beta = T(rz / st->rz);
        if (writer) st->rz_new = rz;
    } else {
        beta = T(st->beta);
        if (writer) st->rz_new = st->rz;
    }
    double contrib = 0.0;
    for (int vb = blockIdx.x; vb < A.nvb; vb += gridDim.x) {
        int row = 0;
        T a[2];
        DirectionOperands<T, CPLX> o{z, p};
        if (!spmv_row_gp<T, CPLX>(A, DirectionGather<T, CPLX>{z, p, beta}, vb, row, a[0], a[1], o)) continue;
#pragma unroll
        for (int w = 0; w < W; w++) {
            const T pk = o.zv[w] + beta * o.pv[w];
            pn[W * row + w] = pk;
            q[W * row + w] = a[w];
            contrib += double(pk) * double(a[w]);
        }
    }
    double v[1] = {contrib};
    partials_write<1>(v, partials + kRowPq * kMaxParts);
}

// npq: partials of p^H q to fold (0: the state holds alpha)
template <typename T, bool CPLX, bool JAC>
__global__ void __launch_bounds__(256) cg_step2(int n, T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                              const T* __restrict__ p, const T* __restrict__ q,
                                              const T* __restrict__ dinv, CgState* st, double* partials, int npq) {
    constexpr int W = CPLX ? 2 : 1;
    const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
    if (st->stop) {
        if (writer) st->done = 1;
        return;
    }
    const double rz_new = st->rz_new;
    T alpha;
    if (npq) {
        double tot[1];
        partials_sum<1>(partials + kRowPq * kMaxParts, npq, tot);
        const double pq = tot[0];
        if (!(pq > 0.0)) {
            if (writer) {
                st->status = (pq == pq) ? MK_ERR_NOT_SPD : MK_ERR_NAN;
                st->done = 1;
            }
            return;
        }
        alpha = T(rz_new / pq);
    } else {
        alpha = T(st->alpha);
    }
    if (writer) st->rz = rz_new;
    double rz = 0.0, rr = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const T d = JAC && dinv ? dinv[i] : T(1);
#pragma unroll
        for (int w = 0; w < W; w++) {
            const int e = W * i + w;
            x[e] += alpha * p[e];
            const T rk = r[e] - alpha * q[e];
            r[e] = rk;
            rr += double(rk) * rk;
            if constexpr (JAC) {
                const T zk = d * rk;
                z[e] = zk;
                rz += double(rk) * zk;
            }
        }
    }
    if constexpr (JAC) {
        double v[2] = {rz, rr};
        partials_write<2>(v, partials);
    } else {
        double v[1] = {rr};
        partials_write<1>(v, partials + kRowRr * kMaxParts);
    }
}

// p^H q -> alpha (launches of more than kFoldParts blocks)
__global__ void __launch_bounds__(1024) cg_alpha_fin(CgState* st, const double* __restrict__ partials, int nparts) {
    if (st->done) return;
    double tot[1];
    partials_sum<1>(partials + kRowPq * kMaxParts, nparts, tot);
    if (threadIdx.x == 0) {
        if (!(tot[0] > 0.0)) { st->status = (tot[0] == tot[0]) ? MK_ERR_NOT_SPD : MK_ERR_NAN; st->done = st->stop = 1; }
        else st->alpha = st->rz_new / tot[0];
    }
}
// rr of the external preconditioner's iteration -> convergence, before the preconditioner runs
__global__ void __launch_bounds__(1024) cg_rr_fin(CgState* st, const double* __restrict__ partials, int nparts) {
    if (st->done) return;
    double tot[1];
    partials_sum<1>(partials + kRowRr * kMaxParts, nparts, tot);
    if (threadIdx.x == 0) {
        st->rr = tot[0];
        st->it += 1;
        if (!(tot[0] == tot[0])) { st->status = MK_ERR_NAN; st->done = 1; }
        else if (tot[0] <= st->tol2 * st->bb) st->done = 1;
    }
}
// the last iteration's rz (Jacobi: and rr) -> rz, beta (and convergence) in the state, for the host
// and for the next batch's first iteration
template <bool JAC>
__global__ void __launch_bounds__(1024) cg_beta_fin(CgState* st, const double* __restrict__ partials, int nparts) {
    if (st->done) return;
    double tot[JAC ? 2 : 1];
    partials_sum<JAC ? 2 : 1>(partials, nparts, tot);
    if (threadIdx.x == 0) {
        const double rz = tot[0];
        if constexpr (JAC) {
            const double rr = tot[1];
            st->rr = rr;
            st->it += 1;
            if (!(rr == rr) || !(rz == rz)) { st->status = MK_ERR_NAN; st->done = 1; }
            else if (rr <= st->tol2 * st->bb) st->done = 1;
        } else if (!(rz > 0.0)) {
            st->status = (rz == rz) ? MK_ERR_NOT_SPD : MK_ERR_NAN;
            st->done = 1;
            return;
        }
        st->beta = rz / st->rz;
        st->rz = rz;
    }
}

// z from an external preconditioner: init, rz
template <typename T, bool CPLX>
__global__ void __launch_bounds__(256) cg_init_z(int n, const T* __restrict__ r, const T* __restrict__ b,
                                               const T* __restrict__ z, T* __restrict__ p, double* partials) {
    double rz = 0.0, rr = 0.0, bb = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if constexpr (CPLX) {
            const T r0 = r[2 * i], r1 = r[2 * i + 1], z0 = z[2 * i], z1 = z[2 * i + 1];
            p[2 * i] = z0; p[2 * i + 1] = z1;
            rz += double(r0) * z0 + double(r1) * z1;
            rr += double(r0) * r0 + double(r1) * r1;
            bb += double(b[2 * i]) * b[2 * i] + double(b[2 * i + 1]) * b[2 * i + 1];
        } else {
            const T r0 = r[i], z0 = z[i];
            p[i] = z0;
            rz += double(r0) * z0;
            rr += double(r0) * r0;
            bb += double(b[i]) * b[i];
        }
    }
    double v[3] = {rz, rr, bb};
    partials_write<3>(v, partials);
}

// rz, rr, bb of the first residual -> the state of a new solve (z from an external preconditioner,
// check_z, must make rz positive)
__global__ void __launch_bounds__(1024) cg_init_fin(CgState* st, const double* __restrict__ partials, int nparts,
                                                    double tol2, int check_z, int* started) {
    double tot[3];
    partials_sum<3>(partials, nparts, tot);
    if (threadIdx.x == 0) {
        st->rz = tot[0];
        st->rr = st->rr0 = tot[1];
        st->bb = tot[2];
        st->tol2 = tol2;
        st->beta = 0.0;
        st->it = 0;
        st->stop = 0;
        st->status = MK_OK;
        st->done = (tot[1] <= tol2 * tot[2]) ? 1 : 0;
        if (!(tot[0] == tot[0]) || !(tot[1] == tot[1])) { st->status = MK_ERR_NAN; st->done = 1; }
        if (check_z && !st->done && !(tot[0] > 0.0)) { st->status = MK_ERR_NOT_SPD; st->done = 1; }
        tell_start(started, st->done);
    }
}

template <typename T, bool CPLX>
__global__ void __launch_bounds__(256) cg_beta(int n, const T* __restrict__ r, const T* __restrict__ z,
                                             const CgState* st, double* partials) {
    if (st->done) return;
    double rz = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if constexpr (CPLX) rz += double(r[2 * i]) * z[2 * i] + double(r[2 * i + 1]) * z[2 * i + 1];
        else rz += double(r[i]) * z[i];
    }
    double v[1] = {rz};
    partials_write<1>(v, partials);
}

// ---------------------------------------------------------------------------------------
// FP64 PCG with an FP32 multigrid preconditioner (vectors as real arrays of len entries;
// complex interleaved gives Re(r^H z) as the plain sum).  The preconditioner runs in FP32,
// so it is not exactly symmetric: beta is the flexible (Polak-Ribiere) form
// beta = r_{k+1}.(z_{k+1} - z_k) / r_k.z_k, with z_k in the other of two FP32 buffers (zold).
// (An FP64 copy of it, written by cgm_spmv and read for m, was 31 MB of an iteration's 1.1 GB on
// 1,310,720 complex rows: 350 us an iteration with it, 342 without.)

// The scalars go through the partials as in cg_step1 / cg_step2 (a = r.z and m = r.zold in rows 0 and
// 1, p^H q in row 2, rr in row 3): folded by the kernel that needs them up to kFoldParts blocks.
static constexpr int kRowUpd = 3;

// x += alpha p ; r -= alpha q ; r32 = float(r) ; rr.  npq: partials of p^H q to fold (0: the state
// holds alpha).
__global__ void __launch_bounds__(256) cgm_update(size_t len, double* __restrict__ x, double* __restrict__ r,
                                                float* __restrict__ r32, const double* __restrict__ p,
                                                const double* __restrict__ q, CgState* st, double* partials, int npq) {
    const int stop = st->stop;
    const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
    // the first element's loads are in flight while alpha is folded
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    double xi = 0.0, ri = 0.0, pi = 0.0, qi = 0.0;
    if (i < len) { xi = x[i]; ri = r[i]; pi = p[i]; qi = q[i]; }
    if (stop) {
        if (writer) st->done = 1;
        return;
    }
    double alpha;
    if (npq) {
        const double rz_new = st->rz_new;
        double tot[1];
        partials_sum<1>(partials + kRowPq * kMaxParts, npq, tot);
        if (!(tot[0] > 0.0)) {
            if (writer) { st->status = (tot[0] == tot[0]) ? MK_ERR_NOT_SPD : MK_ERR_NAN; st->done = 1; }
            return;
        }
        alpha = rz_new / tot[0];
        if (writer) { st->rz = rz_new; st->first = 0; }
    } else {
        alpha = st->alpha;
    }
    double rr = 0.0;
    while (i < len) {
        x[i] = xi + alpha * pi;
        const double rk = ri - alpha * qi;
        r[i] = rk;
        r32[i] = float(rk);
        rr += rk * rk;
        i += stride;
        if (i < len) { xi = x[i]; ri = r[i]; pi = p[i]; qi = q[i]; }
    }
    double v[1] = {rr};
    partials_write<1>(v, partials + kRowUpd * kMaxParts);
}
__global__ void __launch_bounds__(1024) cgm_update_fin(CgState* st, const double* __restrict__ partials, int nparts) {
    if (st->done) return;
    double tot[1];
    partials_sum<1>(partials + kRowUpd * kMaxParts, nparts, tot);
    if (threadIdx.x == 0) {
        st->rr = tot[0];
        st->it += 1;
        if (!(tot[0] == tot[0])) { st->status = MK_ERR_NAN; st->done = 1; }
        else if (tot[0] <= st->tol2 * st->bb) st->done = 1;
    }
}

// beta of the flexible recurrence: a = r.z32, m = r.zold; beta = (a - m) / rz (0 on the first
// iteration); rz = a
__global__ void __launch_bounds__(256) cgm_beta2(size_t len, const double* __restrict__ r,
                                               const float* __restrict__ z32, const float* __restrict__ zold,
                                               const CgState* st, double* partials) {
    if (st->done) return;
    double a = 0.0, m = 0.0;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < len; i += size_t(gridDim.x) * blockDim.x) {
        a += r[i] * double(z32[i]);
        m += r[i] * double(zold[i]);
    }
    double v[2] = {a, m};
    partials_write<2>(v, partials);
}
__global__ void __launch_bounds__(1024) cgm_beta2_fin(CgState* st, const double* __restrict__ partials, int nparts) {
    if (st->done) return;
    double tot[2];
    partials_sum<2>(partials, nparts, tot);
    if (threadIdx.x == 0) {
        if (!(tot[0] > 0.0)) { st->status = (tot[0] == tot[0]) ? MK_ERR_NOT_SPD : MK_ERR_NAN; st->done = 1; }
        else {
            st->beta = st->first ? 0.0 : (tot[0] - tot[1]) / st->rz;
            st->rz = tot[0];
            st->first = 0;
        }
    }
}

// p = z + beta p ; q = A z + beta q (q tracks A p without a second product) ;
// pq = p^H q ; alpha = rz / pq.  z is the FP32 preconditioned residual, A and p, q FP64.
template <bool CPLX>
struct Fp32Gather {
    const float* __restrict__ z;
    __device__ __forceinline__ void operator()(int c, double& xr, double& xi) const {
        if constexpr (CPLX) { xr = double(z[2 * c]); xi = double(z[2 * c + 1]); }
        else { xr = double(z[c]); xi = 0.0; }
    }
};
// the row's own entries of z, p and q, loaded while its gathers are in flight
template <bool CPLX>
struct CgmOperands {
    static constexpr int W = CPLX ? 2 : 1;
    const float* __restrict__ z32;
    const double* __restrict__ p;
    const double* __restrict__ q;
    double zv[W], pv[W], qv[W];
    __device__ __forceinline__ void operator()(int row) {
#pragma unroll
        for (int k = 0; k < W; k++) {
            zv[k] = double(z32[W * row + k]);
            pv[k] = p[W * row + k];
            qv[k] = q[W * row + k];
        }
    }
};
// FOLD: nin partials of a and m to fold, under the first row's loads; otherwise the state holds beta, a
// launch past the end returns before it loads a row, and nothing of the fold is in the row loop: 78
// VGPRs and 6 wavefronts per SIMD (complex; 68 and 7 real) against 87 and 5 (75 and 6), 39.2 us on
// 1,310,720 complex rows of 4 against 45.8 with one kernel for both.
template <bool CPLX, bool FOLD>
__global__ void __launch_bounds__(256) cgm_spmv(SellDev<double> A, const float* __restrict__ z32, double* p, double* q,
                                              CgState* st, double* partials, int nin) {
    const int done = st->done;
    const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
    if (!FOLD && done) {
        if (writer) st->stop = 1;
        return;
    }
    constexpr int W = CPLX ? 2 : 1;
    double beta = FOLD ? 0.0 : st->beta;
    // the state and the first partials are loaded ahead of the row, used behind it
    const double rz = FOLD ? st->rz : 0.0;
    const int first = FOLD ? st->first : 0;
    double pre[2][2];
    if constexpr (FOLD) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = threadIdx.x + u * blockDim.x;
#pragma unroll
            for (int k = 0; k < 2; k++) pre[u][k] = i < nin ? partials[k * kMaxParts + i] : 0.0;
        }
    }
    bool folded = !FOLD;
    double contrib = 0.0;
    for (int vb = blockIdx.x; vb < A.nvb; vb += gridDim.x) {
        int row = 0;
        double a[2];
        CgmOperands<CPLX> o{z32, p, q};
        const bool own = spmv_row_gp<double, CPLX>(A, Fp32Gather<CPLX>{z32}, vb, row, a[0], a[1], o);
        if (FOLD && !folded) {
            if (done) {
                if (writer) st->stop = 1;
                return;
            }
            folded = true;
            double tot[2] = {pre[0][0] + pre[1][0], pre[0][1] + pre[1][1]};
            for (int i = threadIdx.x + 2 * blockDim.x; i < nin; i += blockDim.x) {
                tot[0] += partials[i];
                tot[1] += partials[kMaxParts + i];
            }
            block_sum<2, 1>(tot);
            if (!(tot[0] > 0.0)) {
                if (writer) { st->status = (tot[0] == tot[0]) ? MK_ERR_NOT_SPD : MK_ERR_NAN; st->stop = 1; }
                return;
            }
            beta = first ? 0.0 : (tot[0] - tot[1]) / rz;
            if (writer) st->rz_new = tot[0];  // moved to rz by cgm_update
        }
        if (!own) continue;
#pragma unroll
        for (int k = 0; k < W; k++) {
            const double pk = o.zv[k] + beta * o.pv[k], qk = a[k] + beta * o.qv[k];
            p[W * row + k] = pk;
            q[W * row + k] = qk;
            contrib += pk * qk;
        }
    }
    double v[1] = {contrib};
    partials_write<1>(v, partials + kRowPq * kMaxParts);
}
__global__ void __launch_bounds__(1024) cgm_spmv_fin(CgState* st, const double* __restrict__ partials, int nparts) {
    if (st->done) return;
    double tot[1];
    partials_sum<1>(partials + kRowPq * kMaxParts, nparts, tot);
    if (threadIdx.x == 0) {
        st->pq = tot[0];
        if (!(tot[0] > 0.0)) {
            st->status = (tot[0] == tot[0]) ? MK_ERR_NOT_SPD : MK_ERR_NAN;
            st->done = st->stop = 1;
        } else {
            st->alpha = st->rz / tot[0];
        }
    }
}

// p = q = zold = 0 ; r32 = float(r) ; rr, bb ; state for the first iteration
__global__ void __launch_bounds__(256) cgm_init(size_t len, const double* __restrict__ r, const double* __restrict__ b,
                                              float* __restrict__ r32, double* __restrict__ p, double* __restrict__ q,
                                              float* __restrict__ zold, double* partials) {
    double rr = 0.0, bb = 0.0;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < len; i += size_t(gridDim.x) * blockDim.x) {
        const double ri = r[i], bi = b[i];
        p[i] = 0.0;
        q[i] = 0.0;
        zold[i] = 0.f;
        r32[i] = float(ri);
        rr += ri * ri;
        bb += bi * bi;
    }
    double v[2] = {rr, bb};
    partials_write<2>(v, partials);
}
__global__ void __launch_bounds__(1024) cgm_init_fin(CgState* st, const double* __restrict__ partials, int nparts,
                                                   double tol2, int* started) {
    double tot[2];
    partials_sum<2>(partials, nparts, tot);
    if (threadIdx.x == 0) {
        st->rr = st->rr0 = tot[0];
        st->bb = tot[1];
        st->tol2 = tol2;
        st->rz = 1.0;
        st->it = 0;
        st->stop = 0;
        st->first = 1;
        st->status = MK_OK;
        st->done = (tot[0] <= tol2 * tot[1]) ? 1 : 0;
        if (!(tot[0] == tot[0])) { st->status = MK_ERR_NAN; st->done = 1; }
        tell_start(started, st->done);
    }
}

// ---------------------------------------------------------------------------------------
// misc vector kernels
__global__ void k_axpby(size_t len, double a, const double* x, double b, double* y) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < len) y[i] = a * x[i] + b * y[i];
}
__global__ void k_mass_mul(int n, const double* mass, const double* u, double* b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { b[2 * i] = mass[i] * u[2 * i]; b[2 * i + 1] = mass[i] * u[2 * i + 1]; }
}
__global__ void k_mass_dot(int n, const double* mass, const double* x, double* partials) {
    double c = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) c += mass[i] * (x[2 * i] * x[2 * i] + x[2 * i + 1] * x[2 * i + 1]);
    double v[1] = {c};
    partials_write<1>(v, partials);
}
__global__ void k_dot(size_t len, const double* x, const double* y, double* partials) {
    double c = 0.0;
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < len; i += size_t(gridDim.x) * blockDim.x)
        c += x[i] * y[i];
    double v[1] = {c};
    partials_write<1>(v, partials);
}
__global__ void k_cvt_scaled(size_t len, const double* x, const double* s, float* y) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const double f = 1.0 / sqrt(s[0]);
    if (i < len) y[i] = float(x[i] * f);
}
__global__ void k_add_scaled(size_t len, const float* d, const double* s, double* x) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const double f = sqrt(s[0]);
    if (i < len) x[i] += f * double(d[i]);
}
// ---------------------------------------------------------------------------------------
// host side


// SELL fill: thread (slice s, lane l) writes row order[s C + l] (or s C + l) as column l of
// its slice, entry j at slice_ptr[s] + j C + l; past the row's end a padding entry (its own
// column when that is a valid column, value 0).  VW values per entry (2: complex).  With a
// renumbering the stored row `row` is CSR row rsrc[row] and a CSR column c is stored as
// cmap[c]; a row keeps its entries in CSR order.
template <int VW>
__global__ void __launch_bounds__(256) k_sell_fill(int ns, int C, int n_rows, int m, const int64_t* __restrict__ sptr,
                                                   const int* __restrict__ sw, const int* __restrict__ order,
                                                   const int64_t* __restrict__ rowptr, const int* __restrict__ col,
                                                   const double* __restrict__ val, double scale, int* __restrict__ ocol,
                                                   double* __restrict__ ov64, float* __restrict__ ov32,
                                                   const int* __restrict__ rsrc, const int* __restrict__ cmap) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= int64_t(ns) * C) return;
    const int s = int(t / C), l = int(t - int64_t(s) * C);
    const int r = s * C + l;
    const int row = r < n_rows ? (order ? order[r] : r) : -1;
    const int srow = row >= 0 && rsrc ? rsrc[row] : row;
    const int64_t b = srow >= 0 ? rowptr[srow] : 0;
    const int64_t len = srow >= 0 ? rowptr[srow + 1] - b : 0;
    const int w = sw[s];
    for (int j = 0; j < w; j++) {
        const int64_t e = sptr[s] + int64_t(j) * C + l;
        if (j < len) {
            ocol[e] = cmap ? cmap[col[b + j]] : col[b + j];
#pragma unroll
            for (int q = 0; q < VW; q++) {
                const double v = scale * val[(b + j) * VW + q];
                ov64[e * VW + q] = v;
                ov32[e * VW + q] = float(v);
            }
        } else {
            ocol[e] = (row >= 0 && row < m) ? row : 0;
#pragma unroll
            for (int q = 0; q < VW; q++) { ov64[e * VW + q] = 0.0; ov32[e * VW + q] = 0.0f; }
        }
    }
}

void check_layout(int block, int C, int sigma) {
    MK_CHECK(C > 0 && C % 64 == 0, MK_ERR_ARG, "slice height must be a positive multiple of 64");
    // every SpMV kernel is compiled with __launch_bounds__(256)
    MK_CHECK(block % 64 == 0 && block >= 64 && block <= 256, MK_ERR_ARG, "block_size must be 64, 128 or 256");
    MK_CHECK(sigma >= 1, MK_ERR_ARG, "sigma must be >= 1");
}

void build_sell(mk_op* op, const int64_t* rowptr, const int32_t* col, const double* val, int C, int sigma, double scale,
                const int* rsrc, const int* cmap) {
    const int n = op->n;
    // stored row i is CSR row src(i); a CSR column c is stored as cm(c)
    auto src = [rsrc](int i) { return rsrc ? rsrc[i] : i; };
    auto cm = [cmap](int c) { return cmap ? cmap[c] : c; };
    const int vw = op->cplx ? 2 : 1;
    check_layout(op->block, C, sigma);
    const auto t_start = std::chrono::steady_clock::now();
    auto lap_ms = [&] {
        return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
    };
    // long rows (> max(64, 4 x median length)) go to the wavefront-per-row part
    metriko::HVec<int> lens(static_cast<size_t>(n));
#pragma omp parallel for schedule(static, 65536) if (n > 100000)
    for (int i = 0; i < n; i++) lens[i] = int(rowptr[src(i) + 1] - rowptr[src(i)]);
    // median row length (the element at sorted position n/2) from a length histogram
    int med = 0;
    if (n > 0) {
        constexpr int kHist = 4096;
        std::vector<int64_t> hist(kHist + 1, 0);
#pragma omp parallel if (n > 100000)
        {
            std::vector<int64_t> h(kHist + 1, 0);
#pragma omp for schedule(static, 65536) nowait
            for (int i = 0; i < n; i++) h[size_t(std::min(lens[i], kHist))]++;
#pragma omp critical
            for (int b = 0; b <= kHist; b++) hist[size_t(b)] += h[size_t(b)];
        }
        int64_t cum = 0;
        for (med = 0; med < kHist; med++) {
            cum += hist[size_t(med)];
            if (cum > n / 2) break;
        }
    }
    const int thr = std::max(64, 4 * med);
    // medium rows (more than kMidLen entries) get a group of lanes each instead of one lane;
    // the three classes keep ascending row order (chunked counts, then a parallel fill)
    constexpr int kMidLen = kSellMaxLen;
    auto cls = [&](int i) { return lens[i] > thr ? 2 : lens[i] > kMidLen ? 1 : 0; };
    constexpr int kChunk = 65536;
    const int nch = (n + kChunk - 1) / kChunk;
    std::vector<int> ccount(size_t(nch) * 3, 0);
#pragma omp parallel for schedule(static) if (n > 100000)
    for (int ch = 0; ch < nch; ch++)
        for (int i = ch * kChunk; i < std::min(n, (ch + 1) * kChunk); i++) ccount[size_t(ch) * 3 + cls(i)]++;
    std::vector<int> coff(size_t(nch) * 3, 0);
    int tot3[3] = {0, 0, 0};
    for (int k3 = 0; k3 < 3; k3++)
        for (int ch = 0; ch < nch; ch++) { coff[size_t(ch) * 3 + k3] = tot3[k3]; tot3[k3] += ccount[size_t(ch) * 3 + k3]; }
    metriko::HVec<int> order(static_cast<size_t>(tot3[0]));
    std::vector<int> mrows(static_cast<size_t>(tot3[1])), lrows(static_cast<size_t>(tot3[2]));
#pragma omp parallel for schedule(static) if (n > 100000)
    for (int ch = 0; ch < nch; ch++) {
        int w[3] = {coff[size_t(ch) * 3], coff[size_t(ch) * 3 + 1], coff[size_t(ch) * 3 + 2]};
        for (int i = ch * kChunk; i < std::min(n, (ch + 1) * kChunk); i++) {
            const int k3 = cls(i);
            int* dst = k3 == 0 ? order.data() : k3 == 1 ? mrows.data() : lrows.data();
            dst[w[k3]++] = i;
        }
    }
    const int ns_rows = int(order.size());
    // remaining rows of uneven length: sort inside windows of 1024 rows
    if (sigma <= 1 && ns_rows > 0) {
        int mx = 0;
        int64_t tot = 0;
        for (int r : order) { mx = std::max(mx, lens[r]); tot += lens[r]; }
        if (double(mx) > 2.0 * double(tot) / ns_rows + 8.0) sigma = 1024;
    }
    op->C = C;
    op->sigma = sigma;
    if (sigma > 1) {
#pragma omp parallel for schedule(dynamic, 16) if (ns_rows > 100000)
        for (int w0 = 0; w0 < ns_rows; w0 += sigma) {
            const int w1 = std::min(ns_rows, w0 + sigma);
            std::stable_sort(order.begin() + w0, order.begin() + w1, [&](int a, int b) { return lens[a] > lens[b]; });
        }
    }
    bool permuted = !lrows.empty() || !mrows.empty();
    for (int i = 0; i < ns_rows && !permuted; i++) if (order[i] != i) permuted = true;
    const int n_rows = ns_rows;
    const int ns = (n_rows + C - 1) / C;
    std::vector<int64_t> sptr(size_t(ns) + 1, 0);
    std::vector<int> sw(size_t(ns), 0);
#pragma omp parallel for schedule(static, 1024) if (ns > 10000)
    for (int s = 0; s < ns; s++) {
        int w = 0;
        for (int l = 0; l < C && s * C + l < n_rows; l++) w = std::max<int>(w, lens[order[s * C + l]]);
        sw[s] = w;
    }
    for (int s = 0; s < ns; s++) sptr[s + 1] = sptr[s] + int64_t(sw[s]) * C;
    const int64_t stored = sptr[ns];
    const double t_layout = lap_ms();
    // inverse diagonal (real part) of a square operator; a rectangular one has none
    const bool square = op->m == n;
    metriko::HVec<double> dinv(square ? size_t(n) : 0);
    metriko::HVec<float> dinv32(square ? size_t(n) : 0);
#pragma omp parallel for schedule(static, 4096) if (n > 100000 && square)
    for (int i = 0; i < (square ? n : 0); i++) {
        double d = 0.0;
        const int si = src(i);
        for (int64_t k = rowptr[si]; k < rowptr[si + 1]; k++) if (cm(col[k]) == i) d += scale * val[k * vw];
        dinv[i] = d != 0.0 ? 1.0 / d : 1.0;
        dinv32[i] = float(dinv[i]);
    }
    // medium-row part (CSR, mid_lanes lanes per row: about 4 entries per lane)
    const int nmid = int(mrows.size());
    int mlanes = 4;
    if (nmid) {
        std::vector<int> ml;
        for (int r : mrows) ml.push_back(lens[r]);
        std::nth_element(ml.begin(), ml.begin() + nmid / 2, ml.end());
        const int mm = ml[size_t(nmid / 2)];
        while (mlanes < 16 && mlanes * 4 < mm) mlanes *= 2;
    }
    // medium and long rows as CSR, in their class order (offsets first, then a parallel fill)
    auto fill_csr = [&](const std::vector<int>& rows, std::vector<int64_t>& rp, metriko::HVec<int>& cc,
                        metriko::HVec<double>& cv, metriko::HVec<float>& cv32) {
        const int nr = int(rows.size());
        rp.assign(size_t(nr) + 1, 0);
        for (int w = 0; w < nr; w++) rp[size_t(w) + 1] = rp[size_t(w)] + lens[rows[size_t(w)]];
        const int64_t nz = rp[size_t(nr)];
        cc.resize(size_t(nz));
        cv.resize(size_t(nz) * vw);
        cv32.resize(size_t(nz) * vw);
#pragma omp parallel for schedule(static, 256) if (nz > 200000)
        for (int w = 0; w < nr; w++) {
            const int row = src(rows[size_t(w)]);
            int64_t o = rp[size_t(w)];
            for (int64_t k = rowptr[row]; k < rowptr[row + 1]; k++, o++) {
                cc[size_t(o)] = cm(col[k]);
                for (int c = 0; c < vw; c++) {
                    const double v = scale * val[k * vw + c];
                    cv[size_t(o) * vw + c] = v;
                    cv32[size_t(o) * vw + c] = float(v);
                }
            }
        }
    };
    std::vector<int64_t> mptr;
    metriko::HVec<int> mcol;
    metriko::HVec<double> mval;
    metriko::HVec<float> mval32;
    fill_csr(mrows, mptr, mcol, mval, mval32);
    // long-row part (CSR)
    const int nlong = int(lrows.size());
    std::vector<int64_t> lptr;
    metriko::HVec<int> lcol;
    metriko::HVec<double> lval;
    metriko::HVec<float> lval32;
    fill_csr(lrows, lptr, lcol, lval, lval32);
    // keep every uploaded array non-empty (an operator may consist of long rows only)
    if (sw.empty()) sw.push_back(0);
    if (order.empty()) order.push_back(0);
    const double t_fill = lap_ms();
    hipStream_t st = op->ctx->stream;
    op->nslices = ns;
    op->stored = stored;  // SELL entries only (the long part is long_ptr[nlong] entries)
    op->n_short = n_rows;
    op->nlong = nlong;
    op->slice_ptr.upload(sptr.data(), sptr.size(), st);
    op->slice_w.upload(sw.data(), std::max<size_t>(sw.size(), 1), st);
    const size_t nst = size_t(std::max<int64_t>(stored, 1));
    if (square) {
        op->dinv64.upload(dinv.data(), dinv.size(), st);
        op->dinv32.upload(dinv32.data(), dinv32.size(), st);
    } else {
        op->dinv64.release();
        op->dinv32.release();
    }
    if (permuted) op->perm.upload(order.data(), std::max<size_t>(order.size(), 1), st);
    else op->perm.release();
    // the SELL arrays are filled on the device from the CSR arrays (one upload of the CSR
    // instead of a host fill and an upload of three padded arrays)
    op->col.alloc(nst);
    op->val64.alloc(nst * vw);
    op->val32.alloc(nst * vw);
    if (stored > 0) {
        const int64_t nnz_all = rowptr[n];
        DevBuf<int64_t> drp;
        DevBuf<int> dcol, drs, dcm;
        DevBuf<double> dval;
        if (rsrc) drs.upload(rsrc, size_t(n), st);
        if (cmap) dcm.upload(cmap, size_t(op->m), st);
        drp.upload(rowptr, size_t(n) + 1, st);
        dcol.upload(col, size_t(std::max<int64_t>(nnz_all, 1)), st);
        dval.upload(val, size_t(std::max<int64_t>(nnz_all, 1)) * vw, st);
        const size_t nthr = size_t(ns) * size_t(C);
        const unsigned g = unsigned((nthr + 255) / 256);
        if (vw == 2)
            hipLaunchKernelGGL((k_sell_fill<2>), dim3(g), dim3(256), 0, st, ns, C, n_rows, op->m, op->slice_ptr.p,
                               op->slice_w.p, (const int*)(permuted ? op->perm.p : nullptr), (const int64_t*)drp.p,
                               (const int*)dcol.p, (const double*)dval.p, scale, op->col.p, op->val64.p, op->val32.p,
                               (const int*)drs.p, (const int*)dcm.p);
        else
            hipLaunchKernelGGL((k_sell_fill<1>), dim3(g), dim3(256), 0, st, ns, C, n_rows, op->m, op->slice_ptr.p,
                               op->slice_w.p, (const int*)(permuted ? op->perm.p : nullptr), (const int64_t*)drp.p,
                               (const int*)dcol.p, (const double*)dval.p, scale, op->col.p, op->val64.p, op->val32.p,
                               (const int*)drs.p, (const int*)dcm.p);
        MK_HIP(hipGetLastError());
        MK_HIP(hipStreamSynchronize(st));  // the temporaries are freed on return
    } else {
        MK_HIP(hipMemsetAsync(op->col.p, 0, nst * sizeof(int), st));
        MK_HIP(hipMemsetAsync(op->val64.p, 0, nst * vw * sizeof(double), st));
        MK_HIP(hipMemsetAsync(op->val32.p, 0, nst * vw * sizeof(float), st));
    }
    op->nmid = nmid;
    op->mid_lanes = mlanes;
    if (nmid) {
        op->mid_rows.upload(mrows.data(), mrows.size(), st);
        op->mid_ptr.upload(mptr.data(), mptr.size(), st);
        op->mid_col.upload(mcol.data(), mcol.size(), st);
        op->mid_val64.upload(mval.data(), mval.size(), st);
        op->mid_val32.upload(mval32.data(), mval32.size(), st);
    }
    if (nlong) {
        op->long_rows.upload(lrows.data(), lrows.size(), st);
        op->long_ptr.upload(lptr.data(), lptr.size(), st);
        op->long_col.upload(lcol.data(), lcol.size(), st);
        op->long_val64.upload(lval.data(), lval.size(), st);
        op->long_val32.upload(lval32.data(), lval32.size(), st);
        std::vector<int64_t> sb, se;
        std::vector<int> lsp(size_t(nlong) + 1, 0);
        for (int w = 0; w < nlong; w++) {
            for (int64_t k = lptr[w]; k < lptr[w + 1]; k += kLongSeg) {
                sb.push_back(k);
                se.push_back(std::min<int64_t>(k + kLongSeg, lptr[w + 1]));
            }
            lsp[size_t(w) + 1] = int(sb.size());
        }
        op->nseg = int(sb.size());
        op->seg_beg.upload(sb.data(), std::max<size_t>(sb.size(), 1), st);
        op->seg_end.upload(se.data(), std::max<size_t>(se.size(), 1), st);
        op->lseg_ptr.upload(lsp.data(), lsp.size(), st);
        op->seg_part.alloc(std::max<size_t>(sb.size(), 1) * 64);
    } else {
        op->nseg = 0;
    }
    MK_HIP(hipStreamSynchronize(st));
    if (n > 1000000)
        MK_LOG("[sell] %s %d x %d, %lld stored: layout %.0f ms, fill %.0f ms, upload %.0f ms\n", op->label.c_str(), n,
               op->m, (long long)stored, t_layout, t_fill - t_layout, lap_ms() - t_fill);
    const double sv64 = 8.0 * vw, sv32 = 4.0 * vw;
    const double meta = double(ns) * 12.0 + (permuted ? 4.0 * n : 0.0) + double(nlong + nmid) * 12.0;
    op->bytes64 = double(op->nnz) * (sv64 + 4.0) + meta + double(n) * sv64 * 2.0;
    op->bytes32 = double(op->nnz) * (sv32 + 4.0) + meta + double(n) * sv32 * 2.0;
}


template <typename T>
void spmv_launch(mk_ctx* c, const mk_op* A, const T* val, const T* x, T* y, const T* b, SpmvMode mode, double* out,
                 double bytes, const int* skip) {
    unsigned g = 0;
    const SellDev<T> D = sell_dev<T>(A, val, A->block, &g);
    MK_CHECK(g <= kMaxParts, MK_ERR_ARG, "operator too large for the reduction buffer");
    static const char* kname[] = {"spmv", "spmv_dot", "spmv_resid", "spmv_resid_nored", "spmv_accum"};
    SpmvTimer tm(c, bytes, A, kname[int(mode)], sizeof(T) == 4);
    const unsigned gr = std::max(1u, std::min(g, fin_grid()));  // reducing modes: capped grid
    // the norm alone of a residual is taken between two batches of iterations, whose preconditioned
    // residual's dots wait in rows 0 and 1
    double* part = c->partials.p + (mode == SPMV_RESID && !y ? kRowPq * kMaxParts : 0);
#define MK_SPMV(CPLX, MODE)                                                                                \
    MK_TLAUNCH(tm, 0, (sell_spmv<T, CPLX, MODE>), dim3((MODE == 1 || MODE == 2) ? gr : g), dim3(A->block), 0, \
               c->stream, D, x, y, b, part, skip)
#define MK_SPMV_ALL(CPLX)                            \
    switch (mode) {                                  \
        case SPMV_PLAIN: MK_SPMV(CPLX, 0); break;    \
        case SPMV_DOT: MK_SPMV(CPLX, 1); break;      \
        case SPMV_RESID: MK_SPMV(CPLX, 2); break;    \
        case SPMV_RESID_NORED: MK_SPMV(CPLX, 3); break; \
        case SPMV_ACCUM: MK_SPMV(CPLX, 4); break;    \
    }
    if (A->cplx) { MK_SPMV_ALL(true) } else { MK_SPMV_ALL(false) }
#undef MK_SPMV_ALL
#undef MK_SPMV
    if (mode == SPMV_DOT || mode == SPMV_RESID) finish(c, gr, out, skip, part);
    MK_HIP(hipGetLastError());
}
// One Chebyshev step fused with the residual it needs, row-local:
//   r = b - A x_in ; d = a d + s D^-1 r (first step: d = s D^-1 r) ; x_out = x_in + d.
// The row-local operands of a Chebyshev step (element row of b, x_in, d and the inverse
// diagonal), loaded while the row's gathers are in flight.
template <typename T, bool CPLX>
struct RowOperands {
    static constexpr int W = CPLX ? 2 : 1;
    const T* __restrict__ b;
    const T* __restrict__ x;
    const T* __restrict__ d;   // nullptr: not needed
    const T* __restrict__ dinv;
    T bv[W], xv[W], dv[W], di;
    __device__ __forceinline__ void operator()(int row) {
        di = dinv[row];
#pragma unroll
        for (int q = 0; q < W; q++) {
            bv[q] = b[W * row + q];
            if (x) xv[q] = x[W * row + q];
            dv[q] = d ? d[W * row + q] : T(0);
        }
    }
};

template <typename T, bool CPLX>
__global__ void __launch_bounds__(256) sell_cheb(SellDev<T> A, const T* __restrict__ x_in, T* __restrict__ x_out,
                                               const T* __restrict__ b, T* __restrict__ d,
                                               const T* __restrict__ dinv, T a, T s, int first, const int* skip) {
    if (skip && *skip) return;
    int row = 0;
    T ar, ai;
    RowOperands<T, CPLX> ro{b, x_in, first ? nullptr : d, dinv};
    if (!spmv_row_gp<T, CPLX>(A, PlainGather<T, CPLX>{x_in}, blockIdx.x, row, ar, ai, ro)) return;
    const T sd = s * ro.di;
    if constexpr (CPLX) {
        T d0 = sd * (ro.bv[0] - ar), d1 = sd * (ro.bv[1] - ai);
        if (!first) { d0 += a * ro.dv[0]; d1 += a * ro.dv[1]; }
        d[2 * row] = d0;
        d[2 * row + 1] = d1;
        x_out[2 * row] = ro.xv[0] + d0;
        x_out[2 * row + 1] = ro.xv[1] + d1;
    } else {
        T d0 = sd * (ro.bv[0] - ar);
        if (!first) d0 += a * ro.dv[0];
        d[row] = d0;
        x_out[row] = ro.xv[0] + d0;
    }
}

template <typename T>
void cheb_launch(mk_ctx* c, const mk_op* A, const T* x_in, T* x_out, const T* b, T* d, T a, T s, int first,
                 const int* skip) {
    unsigned g = 0;
    const T* val;
    const T* dinv;
    if constexpr (std::is_same<T, double>::value) { val = A->val64.p; dinv = A->dinv64.p; }
    else { val = A->val32.p; dinv = A->dinv32.p; }
    const SellDev<T> D = sell_dev<T>(A, val, A->block, &g);
    const double vb = double(sizeof(T)) * (A->cplx ? 2 : 1);
    const double bytes = (sizeof(T) == 8 ? A->bytes64 : A->bytes32) + double(A->n) * (vb * (first ? 2.0 : 3.0) +
                                                                                      double(sizeof(T)));
    SpmvTimer tm(c, bytes, A, "cheb", sizeof(T) == 4);
    if (A->cplx)
        MK_TLAUNCH(tm, 0, (sell_cheb<T, true>), dim3(g), dim3(A->block), 0, c->stream, D, x_in, x_out, b, d, dinv,
                   a, s, first, skip);
    else
        MK_TLAUNCH(tm, 0, (sell_cheb<T, false>), dim3(g), dim3(A->block), 0, c->stream, D, x_in, x_out, b, d, dinv,
                   a, s, first, skip);
    MK_HIP(hipGetLastError());
}
template void cheb_launch<double>(mk_ctx*, const mk_op*, const double*, double*, const double*, double*, double,
                                  double, int, const int*);
template void cheb_launch<float>(mk_ctx*, const mk_op*, const float*, float*, const float*, float*, float, float,
                                 int, const int*);

// First two Chebyshev steps from a zero start in one launch: x1 = c0 D^-1 b is formed on the
// fly inside the product (x1 never stored), then r = b - A x1, d = a x1 + s D^-1 r,
// x_out = x1 + d.
template <typename T, bool CPLX>
struct ScaledGather {
    const T* __restrict__ b;
    const T* __restrict__ dinv;
    T c0;
    __device__ __forceinline__ void operator()(int c, T& xr, T& xi) const {
        const T f = c0 * dinv[c];
        if constexpr (CPLX) { xr = f * b[2 * c]; xi = f * b[2 * c + 1]; }
        else { xr = f * b[c]; xi = T(0); }
    }
};
template <typename T, bool CPLX>
__global__ void __launch_bounds__(256) sell_cheb0(SellDev<T> A, const T* __restrict__ b, const T* __restrict__ dinv,
                                                T* __restrict__ x_out, T* __restrict__ d, T c0, T a, T s,
                                                const int* skip) {
    if (skip && *skip) return;
    int row = 0;
    T ar, ai;
    RowOperands<T, CPLX> ro{b, nullptr, nullptr, dinv};
    if (!spmv_row_gp<T, CPLX>(A, ScaledGather<T, CPLX>{b, dinv, c0}, blockIdx.x, row, ar, ai, ro)) return;
    const T di = ro.di, f = c0 * di, sd = s * di;
    if constexpr (CPLX) {
        const T x0 = f * ro.bv[0], x1 = f * ro.bv[1];
        const T d0 = a * x0 + sd * (ro.bv[0] - ar), d1 = a * x1 + sd * (ro.bv[1] - ai);
        d[2 * row] = d0;
        d[2 * row + 1] = d1;
        x_out[2 * row] = x0 + d0;
        x_out[2 * row + 1] = x1 + d1;
    } else {
        const T x0 = f * ro.bv[0];
        const T d0 = a * x0 + sd * (ro.bv[0] - ar);
        d[row] = d0;
        x_out[row] = x0 + d0;
    }
}

template <typename T>
void cheb0_launch(mk_ctx* c, const mk_op* A, const T* b, T* x_out, T* d, T c0, T a, T s, const int* skip) {
    unsigned g = 0;
    const T* val;
    const T* dinv;
    if constexpr (std::is_same<T, double>::value) { val = A->val64.p; dinv = A->dinv64.p; }
    else { val = A->val32.p; dinv = A->dinv32.p; }
    const SellDev<T> D = sell_dev<T>(A, val, A->block, &g);
    const double vb = double(sizeof(T)) * (A->cplx ? 2 : 1);
    const double bytes = (sizeof(T) == 8 ? A->bytes64 : A->bytes32) + double(A->n) * (vb + double(sizeof(T)));
    SpmvTimer tm(c, bytes, A, "cheb0", sizeof(T) == 4);
    if (A->cplx)
        MK_TLAUNCH(tm, 0, (sell_cheb0<T, true>), dim3(g), dim3(A->block), 0, c->stream, D, b, dinv, x_out, d, c0,
                   a, s, skip);
    else
        MK_TLAUNCH(tm, 0, (sell_cheb0<T, false>), dim3(g), dim3(A->block), 0, c->stream, D, b, dinv, x_out, d, c0,
                   a, s, skip);
    MK_HIP(hipGetLastError());
}
template void cheb0_launch<double>(mk_ctx*, const mk_op*, const double*, double*, double*, double, double, double,
                                  const int*);
template void cheb0_launch<float>(mk_ctx*, const mk_op*, const float*, float*, float*, float, float, float,
                                 const int*);

// y = M [u; v] for an operator whose columns [0, m1) act on u and [m1, m) on v (the
// multigrid restriction of a residual: M = [R | -R A], y = R (b - A x) in one launch)
template <typename T, bool CPLX>
struct TwoSourceGather {
    const T* __restrict__ u;
    const T* __restrict__ v;
    int m1;
    __device__ __forceinline__ void operator()(int c, T& xr, T& xi) const {
        const T* s = c < m1 ? u : v;
        const int k = c < m1 ? c : c - m1;
        if constexpr (CPLX) { xr = s[2 * k]; xi = s[2 * k + 1]; }
        else { xr = s[k]; xi = T(0); }
    }
};
// DOTS: also a = r.y and m = r.yold of FP64 vectors r, yold, the dots a flexible PCG needs of its
// preconditioned residual y: partials per block in rows 0 and 1.
template <typename T, bool CPLX>
struct DotOperands {
    static constexpr int W = CPLX ? 2 : 1;
    const double* __restrict__ r;
    const float* __restrict__ yold;
    double rv[W], ov[W];
    __device__ __forceinline__ void operator()(int row) {
#pragma unroll
        for (int q = 0; q < W; q++) { rv[q] = r[W * row + q]; ov[q] = double(yold[W * row + q]); }
    }
};
template <typename T, bool CPLX, bool DOTS>
__global__ void __launch_bounds__(256) sell_spmv2(SellDev<T> A, int m1, const T* __restrict__ u, const T* __restrict__ v,
                                                T* __restrict__ y, const int* skip, const double* __restrict__ r,
                                                const float* __restrict__ yold, double* __restrict__ partials) {
    if (skip && *skip) return;
    int row = 0;
    T a[2];
    if constexpr (!DOTS) {
        if (!spmv_row_g<T, CPLX>(A, TwoSourceGather<T, CPLX>{u, v, m1}, blockIdx.x, row, a[0], a[1])) return;
        if constexpr (CPLX) { y[2 * row] = a[0]; y[2 * row + 1] = a[1]; }
        else y[row] = a[0];
    } else {
        constexpr int W = CPLX ? 2 : 1;
        DotOperands<T, CPLX> o{r, yold};
        double d[2] = {0.0, 0.0};
        if (spmv_row_gp<T, CPLX>(A, TwoSourceGather<T, CPLX>{u, v, m1}, blockIdx.x, row, a[0], a[1], o)) {
#pragma unroll
            for (int q = 0; q < W; q++) {
                y[W * row + q] = a[q];
                d[0] += o.rv[q] * double(a[q]);
                d[1] += o.rv[q] * o.ov[q];
            }
        }
        partials_write<2>(d, partials);
    }
}

// r (with yold and partials): the dots too; returns the number of partials
template <typename T>
unsigned spmv2_launch(mk_ctx* c, const mk_op* A, int m1, const T* u, const T* v, T* y, const int* skip, const char* name,
                      const double* r, const float* yold, double* partials) {
    unsigned g = 0;
    const T* val;
    if constexpr (std::is_same<T, double>::value) val = A->val64.p;
    else val = A->val32.p;
    const SellDev<T> D = sell_dev<T>(A, val, A->block, &g);
    MK_CHECK(!r || g <= kMaxParts, MK_ERR_ARG, "operator too large for the reduction buffer");
    SpmvTimer tm(c, sizeof(T) == 8 ? A->bytes64 : A->bytes32, A, name, sizeof(T) == 4);
#define MK_SPMV2(CP, DOTS)                                                                                        \
    MK_TLAUNCH(tm, 0, (sell_spmv2<T, CP, DOTS>), dim3(g), dim3(A->block), 0, c->stream, D, m1, u, v, y, skip, r, \
               yold, partials)
    constexpr bool dots = std::is_same<T, float>::value;  // only the FP32 V-cycle is asked for them
    MK_CHECK(dots || !r, MK_ERR_UNSUPPORTED, "two-source product: dots in FP32 only");
    if (A->cplx) { if (r) MK_SPMV2(true, dots); else MK_SPMV2(true, false); }
    else { if (r) MK_SPMV2(false, dots); else MK_SPMV2(false, false); }
#undef MK_SPMV2
    MK_HIP(hipGetLastError());
    return g;
}
template unsigned spmv2_launch<double>(mk_ctx*, const mk_op*, int, const double*, const double*, double*, const int*,
                                       const char*, const double*, const float*, double*);
template unsigned spmv2_launch<float>(mk_ctx*, const mk_op*, int, const float*, const float*, float*, const int*,
                                      const char*, const double*, const float*, double*);

template <typename T>
__global__ void k_copy(size_t len, const T* __restrict__ x, T* __restrict__ y, const int* skip) {
    if (skip && *skip) return;
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < len) y[i] = x[i];
}
template <typename T>
void copy_launch(mk_ctx* c, size_t len, const T* x, T* y, const int* skip) {
    hipLaunchKernelGGL(k_copy<T>, dim3(blocks_for(len)), dim3(256), 0, c->stream, len, x, y, skip);
}
template void copy_launch<double>(mk_ctx*, size_t, const double*, double*, const int*);
template void copy_launch<float>(mk_ctx*, size_t, const float*, float*, const int*);

template void spmv_launch<double>(mk_ctx*, const mk_op*, const double*, const double*, double*, const double*,
                                  SpmvMode, double*, double, const int*);
template void spmv_launch<float>(mk_ctx*, const mk_op*, const float*, const float*, float*, const float*, SpmvMode,
                                 double*, double, const int*);

void spmv64(mk_ctx* c, const mk_op* A, const double* x, double* y, const double* b, SpmvMode mode, double* out,
            int*) {
    const double extra = (mode == SPMV_RESID || mode == SPMV_RESID_NORED || mode == SPMV_ACCUM)
                             ? A->n * 8.0 * (A->cplx ? 2 : 1) : 0.0;
    spmv_launch<double>(c, A, A->val64.p, x, y, b, mode, out, A->bytes64 + extra, nullptr);
}
void spmv32(mk_ctx* c, const mk_op* A, const float* x, float* y, SpmvMode mode, double* out, int*) {
    spmv_launch<float>(c, A, A->val32.p, x, y, nullptr, mode, out, A->bytes32, nullptr);
}

void axpby64(mk_ctx* c, size_t len, double a, const double* x, double b, double* y) {
    hipLaunchKernelGGL(k_axpby, dim3(blocks_for(len)), dim3(256), 0, c->stream, len, a, x, b, y);
    MK_HIP(hipGetLastError());
}
void dot64(mk_ctx* c, size_t len, const double* x, const double* y, double* out_dev) {
    const unsigned g = fgrid(len);
    hipLaunchKernelGGL(k_dot, dim3(g), dim3(256), 0, c->stream, len, x, y, c->partials.p);
    finish(c, g, out_dev);
    MK_HIP(hipGetLastError());
}
void mass_mul(mk_ctx* c, int n, const double* mass, const double* u, double* b) {
    hipLaunchKernelGGL(k_mass_mul, dim3(blocks_for(n)), dim3(256), 0, c->stream, n, mass, u, b);
    MK_HIP(hipGetLastError());
}
void mass_dot(mk_ctx* c, int n, const double* mass, const double* x, double* out_dev) {
    const unsigned g = fgrid(size_t(n));
    hipLaunchKernelGGL(k_mass_dot, dim3(g), dim3(256), 0, c->stream, n, mass, x, c->partials.p);
    finish(c, g, out_dev);
    MK_HIP(hipGetLastError());
}
void cvt64to32_scaled(mk_ctx* c, size_t len, const double* x, const double* s_dev, float* y) {
    hipLaunchKernelGGL(k_cvt_scaled, dim3(blocks_for(len)), dim3(256), 0, c->stream, len, x, s_dev, y);
    MK_HIP(hipGetLastError());
}
void add32to64_scaled(mk_ctx* c, size_t len, const float* d, const double* s_dev, double* x) {
    hipLaunchKernelGGL(k_add_scaled, dim3(blocks_for(len)), dim3(256), 0, c->stream, len, d, s_dev, x);
    MK_HIP(hipGetLastError());
}

// Generic PCG on the device.
static inline void mg_apply(mk_ctx* c, Mg* g, const double* b, double* x, const int* skip, bool) {
    mg_apply64(c, g, b, x, skip);
}
static inline void mg_apply(mk_ctx* c, Mg* g, const float* b, float* x, const int* skip, bool drop) {
    mg_apply32(c, g, b, x, skip, drop);
}

// Runs body(batch) on the context stream: eagerly, or -- when graphs are on and timing is off -- by
// replaying a hipGraph captured from the same call the first time this key is seen.  It must only launch kernels on
// c->stream whose arguments are fixed by the key: the context (its id and its partials, state
// and scalar buffers), the hierarchy (its id: its level buffers live as long as it does) and
// the solve's vectors and value arrays (`buffers`).  The graphs are cached on the operator, so
// an operator is only ever run on the context it was created on.
template <typename F>
static void run_batch(mk_ctx* c, const mk_op* A_, const Mg* mg, std::vector<uintptr_t> buffers, int batch, F&& body) {
    mk_op* A = const_cast<mk_op*>(A_);
    MK_CHECK(A->ctx == c, MK_ERR_ARG, "operator used with a context other than the one it was created on");
    if (!c->use_graphs || c->time_spmv) {
        body(batch);
        c->eager_batches++;
        return;
    }
    GraphKeyParts kp;
    kp.ctx_uid = c->uid;
    kp.mg_uid = mg_uid(mg);
    kp.state = uintptr_t(c->state.p);
    kp.partials = uintptr_t(c->partials.p);
    kp.scal = uintptr_t(c->scal.p);
    kp.buffers = std::move(buffers);
    kp.batch = batch;
    const std::vector<uintptr_t> key = make_graph_key(kp);
    mk_op::Graph* G = nullptr;
    for (auto& g : A->graphs) if (g.key == key) { G = &g; break; }
    if (!G) {
        if (A->graphs.size() >= 16) {  // bounded cache: drop the oldest
            if (A->graphs.front().exec) MK_HIP(hipGraphExecDestroy(A->graphs.front().exec));
            A->graphs.erase(A->graphs.begin());
        }
        const int64_t calls0 = c->spmv_calls;
        const double bytes0 = c->spmv_bytes;
        const auto t_cap = std::chrono::steady_clock::now();
        MK_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeRelaxed));
        hipGraph_t graph = nullptr;
        try {
            body(batch);
        } catch (...) {
            (void)hipStreamEndCapture(c->stream, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        MK_HIP(hipStreamEndCapture(c->stream, &graph));
        mk_op::Graph ng;
        ng.key = key;
        hipError_t e = hipGraphInstantiate(&ng.exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (e != hipSuccess) throw Error(MK_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        ng.spmv_calls = c->spmv_calls - calls0;
        ng.spmv_bytes = c->spmv_bytes - bytes0;
        c->spmv_calls = calls0;
        c->spmv_bytes = bytes0;
        A->graphs.push_back(std::move(ng));
        G = &A->graphs.back();
        c->graph_captures++;
        MK_LOG("[graph] %s: %d iterations captured and instantiated in %.1f ms\n", A->label.c_str(), batch,
               std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_cap).count());
    }
    MK_HIP(hipGraphLaunch(G->exec, c->stream));
    c->spmv_calls += G->spmv_calls;
    c->spmv_bytes += G->spmv_bytes;
    c->graph_replays++;
}

// m iterations as captured batches: whole check intervals, then power-of-two pieces (a few
// graph sizes per operator, each captured once and replayed by every later solve)
template <typename F>
static void run_batches(int m, int interval, F&& batch) {
    for (; interval > 0 && m >= interval; m -= interval) batch(interval);
    for (int p = 1 << 30; m > 0; p >>= 1)
        if (p <= m) { batch(p); m -= p; }
}

// Runs a started solve (its state on the device): launch(m) queues m iterations; resid() queues
// the true residual of x into the state behind a batch that is expected to be the last, so that a
// solve that ends where its operator's last one did costs one round trip to the host.
template <typename L, typename R>
static CgResult drive(mk_ctx* c, int hint, int maxiter, int check_every, bool captured, L&& launch, R&& resid) {
    BatchPlanner plan(c->time_spmv ? 1 : check_every);
    CgState* h = static_cast<CgState*>(c->pin);
    static_assert(sizeof(CgState) <= mk_ctx::kPinBytes, "CgState does not fit the readback memory");
    int launched = 0, batch = plan.first(hint);
    for (;;) {
        batch = std::min(batch, maxiter - launched);
        if (launched == 0 && batch > 2) {
            const int p = BatchPlanner::before_start(batch, captured);
            launch(p);
            launched += p;
            batch = start_converged(c) ? 0 : batch - p;
        }
        if (batch > 0) { launch(batch); launched += batch; }
        const bool checked = plan.last && !c->time_spmv && resid();
        MK_HIP(hipGetLastError());
        MK_HIP(hipMemcpyAsync(h, c->state.p, sizeof(CgState), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipStreamSynchronize(c->stream));
        timing_flush(c);
        if (h->done || h->it >= maxiter) {
            CgResult res{h->status, h->it, h->rr, h->bb, checked ? h->true_rr : -1.0};
            if (res.status == MK_OK && !h->done) res.status = MK_ERR_NO_CONVERGENCE;
            return res;
        }
        batch = plan.next(h->it, h->rr, h->rr0, h->tol2 * h->bb);
    }
}

// PCG on r (the initial residual); b for its norm.  resid as in drive().
template <typename T, typename R>
static CgResult cg_run(mk_ctx* c, const mk_op* A, const T* val, const T* dinv, const T* b, T* x, T* r, T* z, T* p, T* p2,
                       T* q, double rel_tol, int hint, int maxiter, int check_every, double bytes, Mg* mg, bool drop, R&& resid) {
    const int n = A->n;
    const size_t len = size_t(n) * (A->cplx ? 2 : 1);
    const unsigned g = blocks_for(n);
    MK_CHECK(g <= kMaxParts, MK_ERR_ARG, "operator too large for the reduction buffer");
    CgState* st = c->state.p;
    const unsigned gn = fgrid(size_t(n));
    if (mg) {
        mg_apply(c, mg, r, z, nullptr, drop);
        if (A->cplx)
            hipLaunchKernelGGL((cg_init_z<T, true>), dim3(gn), dim3(256), 0, c->stream, n, r, b, z, p, c->partials.p);
        else
            hipLaunchKernelGGL((cg_init_z<T, false>), dim3(gn), dim3(256), 0, c->stream, n, r, b, z, p, c->partials.p);
    } else {
        if (A->cplx)
            hipLaunchKernelGGL((cg_init<T, true>), dim3(gn), dim3(256), 0, c->stream, n, r, b, dinv, z, p,
                               c->partials.p);
        else
            hipLaunchKernelGGL((cg_init<T, false>), dim3(gn), dim3(256), 0, c->stream, n, r, b, dinv, z, p,
                               c->partials.p);
    }
    hipLaunchKernelGGL(cg_init_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)c->partials.p, int(gn),
                       rel_tol * rel_tol, mg ? 1 : 0, arm_start(c));
    MK_HIP(hipGetLastError());
    unsigned gs = 0;
    const SellDev<T> D = sell_dev<T>(A, val, A->block, &gs);
    const unsigned gr = std::max(1u, std::min(gs, fin_grid()));
    const bool fold = std::max(gr, gn) <= kFoldParts;
    double* part = c->partials.p;
    // `batch` iterations from direction buffer pa (the other one: pb), which alternate
    auto iterations = [&](int batch, T* pa, T* pb) {
        for (int k = 0; k < batch; k++, std::swap(pa, pb)) {
            const int nin = fold && k ? int(gn) : 0;
            {
                SpmvTimer tm(c, bytes, A, "cg_spmv", sizeof(T) == 4);
#define MK_STEP1(CP, JAC)                                                                                               \
    MK_TLAUNCH(tm, 0, (cg_step1<T, CP, JAC>), dim3(gr), dim3(A->block), 0, c->stream, D, (const T*)z, (const T*)pa, pb, \
               q, st, part, nin)
                if (A->cplx) { if (mg) MK_STEP1(true, false); else MK_STEP1(true, true); }
                else { if (mg) MK_STEP1(false, false); else MK_STEP1(false, true); }
#undef MK_STEP1
            }
            if (!fold) hipLaunchKernelGGL(cg_alpha_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)part, int(gr));
            const int npq = fold ? int(gr) : 0;
#define MK_STEP2(CP, JAC)                                                                                       \
    hipLaunchKernelGGL((cg_step2<T, CP, JAC>), dim3(gn), dim3(256), 0, c->stream, n, x, r, z, (const T*)pb, \
                       (const T*)q, dinv, st, part, npq)
            if (A->cplx) { if (mg) MK_STEP2(true, false); else MK_STEP2(true, true); }
            else { if (mg) MK_STEP2(false, false); else MK_STEP2(false, true); }
#undef MK_STEP2
            if (mg) {
                hipLaunchKernelGGL(cg_rr_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)part, int(gn));
                mg_apply(c, mg, r, z, &st->done, drop);
                if (A->cplx)
                    hipLaunchKernelGGL((cg_beta<T, true>), dim3(gn), dim3(256), 0, c->stream, n, r, z, (const CgState*)st,
                                       part);
                else
                    hipLaunchKernelGGL((cg_beta<T, false>), dim3(gn), dim3(256), 0, c->stream, n, r, z,
                                       (const CgState*)st, part);
            }
            if (fold && k + 1 < batch) continue;
            // as many threads as the fold has, so the order of the sum, and with it every bit of the
            // solution, does not depend on where a batch ends
            const dim3 nt(fold ? A->block : 1024);
            if (mg) hipLaunchKernelGGL((cg_beta_fin<false>), dim3(1), nt, 0, c->stream, st, (const double*)part, int(gn));
            else hipLaunchKernelGGL((cg_beta_fin<true>), dim3(1), nt, 0, c->stream, st, (const double*)part, int(gn));
        }
    };
    return drive(c, hint, maxiter, check_every, mg != nullptr, [&](int batch) {
        if (!mg) {
            iterations(batch, p, p2);
            if (batch & 1) std::swap(p, p2);
            return;
        }
        run_batches(batch, check_every, [&](int m) {
            run_batch(c, A, mg, {uintptr_t(sizeof(T)), uintptr_t(val), uintptr_t(x), uintptr_t(r), uintptr_t(z), uintptr_t(p),
                                 uintptr_t(p2), uintptr_t(q), uintptr_t(drop)},
                      m, [&](int k) { iterations(k, p, p2); });
            if (m & 1) std::swap(p, p2);
        });
    }, resid);
}

// ||b - A x||^2 into the CG state, for drive()
static auto true_residual(mk_ctx* c, const mk_op* A, const double* b, const double* x) {
    return [=] {
        spmv64(c, A, x, nullptr, b, SPMV_RESID, &c->state.p->true_rr, nullptr);
        return true;
    };
}

CgResult cg64(mk_ctx* c, const mk_op* A, const double* b, double* x, double rel_tol, int hint, int maxiter, bool jacobi,
              int check_every, Mg* mg) {
    Work& w = work(c);
    const size_t len = size_t(A->n) * (A->cplx ? 2 : 1);
    w.r.ensure(len); w.z.ensure(len); w.p.ensure(len); w.p2.ensure(len); w.q.ensure(len);
    spmv64(c, A, x, w.r.p, b, SPMV_RESID_NORED, nullptr, nullptr);
    return cg_run<double>(c, A, A->val64.p, jacobi ? A->dinv64.p : nullptr, b, x, w.r.p, w.z.p, w.p.p, w.p2.p, w.q.p, rel_tol,
                          hint, maxiter, check_every, A->bytes64, mg, false, true_residual(c, A, b, x));
}

// x = A^-1 b from zero in FP32 (drop: see mg_drop_fp32_null)
CgResult cg32(mk_ctx* c, const mk_op* A, const float* b, float* x, double rel_tol, int maxiter, bool jacobi,
              int check_every, Mg* mg, bool drop) {
    Work& w = work(c);
    const size_t len = size_t(A->n) * (A->cplx ? 2 : 1);
    w.r32.ensure(len); w.z32.ensure(len); w.p32.ensure(len); w.p2_32.ensure(len); w.q32.ensure(len);
    MK_HIP(hipMemsetAsync(x, 0, len * sizeof(float), c->stream));
    MK_HIP(hipMemcpyAsync(w.r32.p, b, len * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
    return cg_run<float>(c, A, A->val32.p, jacobi ? A->dinv32.p : nullptr, b, x, w.r32.p, w.z32.p, w.p32.p, w.p2_32.p, w.q32.p,
                         rel_tol, 0, maxiter, check_every, A->bytes32, mg, drop, [] { return false; });
}

// FP64 flexible PCG whose multigrid V-cycle runs in FP32 (vectors converted at its ends).
CgResult cg64_mg32(mk_ctx* c, const mk_op* A, const double* b, double* x, double rel_tol, int hint, int maxiter,
                   int check_every, Mg* mg) {
    Work& w = work(c);
    const size_t len = size_t(A->n) * (A->cplx ? 2 : 1);
    w.r.ensure(len); w.p.ensure(len); w.q.ensure(len);
    w.r32.ensure(len); w.z32.ensure(len); w.z2_32.ensure(len);
    float *zc = w.z32.p, *zo = w.z2_32.p;  // the V-cycle's current output and the previous one
    MK_CHECK(blocks_for(len) <= kMaxParts, MK_ERR_ARG, "operator too large for the reduction buffer");
    spmv64(c, A, x, w.r.p, b, SPMV_RESID_NORED, nullptr, nullptr);
    CgState* st = c->state.p;
    const unsigned gl = fgrid(len);
    hipLaunchKernelGGL(cgm_init, dim3(gl), dim3(256), 0, c->stream, len, (const double*)w.r.p, b, w.r32.p, w.p.p, w.q.p,
                       zo, c->partials.p);
    hipLaunchKernelGGL(cgm_init_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)c->partials.p, int(gl),
                       rel_tol * rel_tol, arm_start(c));
    double* part = c->partials.p;
    // the V-cycle on r32 and the two dots beta needs, in its last kernel where that can; returns
    // their partials
    auto precondition = [&](float* z, const float* zold) {
        const unsigned np = mg_apply32_dots(c, mg, w.r32.p, z, &st->done, w.r.p, zold, part);
        if (np) return np;
        hipLaunchKernelGGL(cgm_beta2, dim3(gl), dim3(256), 0, c->stream, len, (const double*)w.r.p,
                           (const float*)z, zold, (const CgState*)st, part);
        return gl;
    };
    const unsigned gb = precondition(zc, zo);
    MK_HIP(hipGetLastError());
    unsigned gs = 0;
    const SellDev<double> D = sell_dev<double>(A, A->val64.p, A->block, &gs);
    const unsigned gsr = std::max(1u, std::min(gs, fin_grid()));
    const bool fold_b = gb <= kFoldParts && gsr <= kFoldParts;
    // one iteration: beta, p/q update with A z (fused), x/r update, V-cycle on the new residual
    auto iteration = [&](const float* z, float* zn) {
        if (!fold_b)
            hipLaunchKernelGGL(cgm_beta2_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)part, int(gb));
        const int nin = fold_b ? int(gb) : 0;
        {
            SpmvTimer tm(c, A->bytes64 + double(len) * (4.0 + 8.0 * 4.0), A, "cg_spmv", false);
#define MK_CGM(CP, FOLD) \
    MK_TLAUNCH(tm, 0, (cgm_spmv<CP, FOLD>), dim3(gsr), dim3(A->block), 0, c->stream, D, z, w.p.p, w.q.p, st, part, nin)
            if (A->cplx) { if (fold_b) MK_CGM(true, true); else MK_CGM(true, false); }
            else { if (fold_b) MK_CGM(false, true); else MK_CGM(false, false); }
#undef MK_CGM
        }
        if (!fold_b)
            hipLaunchKernelGGL(cgm_spmv_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)part, int(gsr));
        hipLaunchKernelGGL(cgm_update, dim3(gl), dim3(256), 0, c->stream, len, x, w.r.p, w.r32.p,
                           (const double*)w.p.p, (const double*)w.q.p, st, part, fold_b ? int(gsr) : 0);
        hipLaunchKernelGGL(cgm_update_fin, dim3(1), dim3(1024), 0, c->stream, st, (const double*)part, int(gl));
        precondition(zn, z);
    };
    return drive(c, hint, maxiter, check_every, true, [&](int batch) {
        run_batches(batch, check_every, [&](int m) {
            run_batch(c, A, mg, {uintptr_t(4), uintptr_t(A->val64.p), uintptr_t(x), uintptr_t(w.r.p),
                                 uintptr_t(w.r32.p), uintptr_t(zc), uintptr_t(zo), uintptr_t(w.p.p),
                                 uintptr_t(w.q.p)},
                      m, [&](int k) {
                          float *a = zc, *b2 = zo;
                          for (; k > 0; k--, std::swap(a, b2)) iteration(a, b2);
                      });
            if (m & 1) std::swap(zc, zo);
        });
    }, true_residual(c, A, b, x));
}

// Iterative refinement: FP64 residual r = b - A x, FP32 PCG correction on r/||r||.
SolveResult solve_spd(mk_ctx* c, const mk_op* A, const double* b, double* x, const mk_solve_opts& o, Mg* pre,
                      double target) {
    MK_CHECK(o.precision >= MK_PREC_FP64 && o.precision <= MK_PREC_MIXED_MG, MK_ERR_ARG, "unknown precision mode");
    // goal: where the iteration stops; o.tol: what the result must meet (a goal below the FP64
    // floor eps ||A|| ||x|| / ||b|| of the true residual is met as far as that floor allows)
    const double goal = (target > 0.0 && target < o.tol) ? target : o.tol;
    const bool jac = o.precond == MK_PRECOND_JACOBI;
    Mg* mg = (o.precond == MK_PRECOND_AMG) ? (pre ? pre : A->mg) : nullptr;
    MK_CHECK(o.precond != MK_PRECOND_AMG || mg, MK_ERR_ARG, "AMG preconditioner requested but not built");
    SolveResult res{MK_OK, 0, 0, 0.0};
    const size_t len = size_t(A->n) * (A->cplx ? 2 : 1);
    // FP32 multigrid inside FP64 PCG; without multigrid there is no FP32 work to do: plain FP64
    const bool mg32 = o.precision == MK_PREC_MIXED_MG && mg;
    if (o.precision == MK_PREC_FP64 || o.precision == MK_PREC_MIXED_MG) {
        // the recurrences can drift from the true residual: it is recomputed in FP64 and the
        // solve restarts from x (at most twice) while it is above the tolerance
        for (int attempt = 0;; attempt++) {
            const int hint = attempt == 0 ? A->last_iters : 0;
            const CgResult cr = mg32 ? cg64_mg32(c, A, b, x, goal, hint, o.maxiter - res.iters, o.check_every, mg)
                                     : cg64(c, A, b, x, goal, hint, o.maxiter - res.iters, jac, o.check_every, mg);
            res.iters += cr.iters;
            double rr = cr.true_rr;
            if (!(rr >= 0.0)) {
                true_residual(c, A, b, x)();
                double* h = static_cast<double*>(c->pin);
                MK_HIP(hipMemcpyAsync(h, &c->state.p->true_rr, sizeof(double), hipMemcpyDeviceToHost, c->stream));
                MK_HIP(hipStreamSynchronize(c->stream));
                rr = *h;
            }
            res.rel_residual = cr.bb > 0 ? std::sqrt(rr / cr.bb) : std::sqrt(rr);
            res.status = cr.status;
            if (res.status == MK_ERR_NO_CONVERGENCE && res.rel_residual <= o.tol) res.status = MK_OK;
            if (!(res.status == MK_OK && res.rel_residual > o.tol && attempt < 2 && res.iters < o.maxiter))
                break;
            res.refinements++;
        }
        A->last_iters = res.iters;
        if (res.status == MK_OK && res.rel_residual > o.tol) res.status = MK_ERR_NO_CONVERGENCE;
        return res;
    }
    Work& w = work(c);
    w.t.ensure(len); w.r32.ensure(len); w.x32.ensure(len);
    double* bb = c->scal.p + 4;
    double* rr = c->scal.p + 5;
    dot64(c, len, b, b, bb);
    double hbb = 0.0;
    MK_HIP(hipMemcpyAsync(&hbb, bb, sizeof(double), hipMemcpyDeviceToHost, c->stream));
    MK_HIP(hipStreamSynchronize(c->stream));
    if (hbb == 0.0) {
        MK_HIP(hipMemsetAsync(x, 0, len * sizeof(double), c->stream));
        MK_HIP(hipStreamSynchronize(c->stream));
        return res;
    }
    double prev = HUGE_VAL;
    int stagn = 0;
    bool drop = false;
    // the FP32 work vectors used by cg32 are r32,z32,p32,q32; the normalised rhs lives in x32's twin
    DevBuf<float>& rhs32 = w.x32;
    DevBuf<float>& d32 = w.d32;
    d32.ensure(len);
    for (;;) {
        spmv64(c, A, x, w.t.p, b, SPMV_RESID, rr, nullptr);
        double hrr = 0.0;
        MK_HIP(hipMemcpyAsync(&hrr, rr, sizeof(double), hipMemcpyDeviceToHost, c->stream));
        MK_HIP(hipStreamSynchronize(c->stream));
        const double rel = std::sqrt(hrr / hbb);
        res.rel_residual = rel;
        if (!(rel == rel)) { res.status = MK_ERR_NAN; break; }
        if (rel <= goal) break;
        if (res.refinements >= o.max_refine) { res.status = rel <= o.tol ? MK_OK : MK_ERR_NO_CONVERGENCE; break; }
        if (rel > 0.5 * prev) { if (++stagn >= 3) { res.status = rel <= o.tol ? MK_OK : MK_ERR_STAGNATION; break; } }
        else stagn = 0;
        prev = rel;
        cvt64to32_scaled(c, len, w.t.p, rr, rhs32.p);
        const double itol = std::max(o.inner_tol, 0.5 * goal / rel);
        CgResult cr = cg32(c, A, rhs32.p, d32.p, std::min(itol, 0.5), o.maxiter - res.iters, jac, o.check_every, mg, drop);
        // An operator that is singular in FP32 breaks down along the direction that the hierarchy's coarsest
        // inverse, formed in FP64, still resolves: the corrections go on without it.
        if ((cr.status == MK_ERR_NOT_SPD || cr.status == MK_ERR_NAN) && mg && !drop && mg_drop_fp32_null(c, mg)) {
            res.iters += cr.iters;
            drop = true;
            cr = cg32(c, A, rhs32.p, d32.p, std::min(itol, 0.5), o.maxiter - res.iters, jac, o.check_every, mg, drop);
        }
        res.iters += cr.iters;
        res.refinements++;
        if (cr.status == MK_ERR_NOT_SPD || cr.status == MK_ERR_NAN) { res.status = cr.status; break; }
        add32to64_scaled(c, len, d32.p, rr, x);
        if (res.iters >= o.maxiter) {
            spmv64(c, A, x, w.t.p, b, SPMV_RESID, rr, nullptr);
            MK_HIP(hipMemcpyAsync(&hrr, rr, sizeof(double), hipMemcpyDeviceToHost, c->stream));
            MK_HIP(hipStreamSynchronize(c->stream));
            res.rel_residual = std::sqrt(hrr / hbb);
            if (res.rel_residual > o.tol) res.status = MK_ERR_NO_CONVERGENCE;
            break;
        }
    }
    return res;
}

}  // namespace mk
