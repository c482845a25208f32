// Dense inverse of the coarsest multigrid operator, built and applied on the device.
//
// The inverse of a Hermitian positive definite n x n matrix is formed in place by blocked
// Gauss-Jordan elimination without pivoting (its pivots are the Cholesky pivots): per block of
// kNb columns one kernel inverts the diagonal block and forms the pivot rows, one updates the
// whole matrix by a rank-kNb product on the FP64 matrix cores.  Matrices are row-major with
// leading dimension ld = n rounded up to kTile, padded with the identity.
//
// Everything is FP64 and stays FP64 when it is applied to FP32 vectors: rounding the inverse of
// an operator of condition 1e7 and more to FP32 can make it indefinite, and the size limit below
// costs no more in FP64 than a smoothed level does.
#include "mk_internal.h"
#include "sell.h"

namespace mk {

namespace {

constexpr int kNb = 32;    // columns eliminated per step
constexpr int kTile = 64;  // tile of the rank-kNb update (and of the padding)

typedef double d4 __attribute__((ext_vector_type(4)));

// v_mfma_f64_16x16x4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and, in element r of the
// result, D[l / 16 + 4 r][l % 16].
__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Row `blockIdx.x` of the padded matrix from the CSR operator, and the row's diagonal (which
// scales the guard of a pivot that rounding makes non-positive).
template <bool CPLX>
__global__ void __launch_bounds__(256) k_dense_fill(int n, int ld, const int64_t* __restrict__ ptr,
                                                    const int* __restrict__ col, const double* __restrict__ val,
                                                    double* __restrict__ A, double* __restrict__ diag) {
    constexpr int W = CPLX ? 2 : 1;
    const int i = blockIdx.x;
    double* row = A + size_t(i) * ld * W;
    for (int j = threadIdx.x; j < ld * W; j += 256) row[j] = 0.0;
    if (threadIdx.x == 0) diag[i] = i < n ? 0.0 : 1.0;
    __syncthreads();
    if (i >= n) {
        if (threadIdx.x == 0) row[size_t(i) * W] = 1.0;
        return;
    }
    for (int64_t k = ptr[i] + threadIdx.x; k < ptr[i + 1]; k += 256) {
        const int c = col[k];
        for (int q = 0; q < W; q++) row[size_t(c) * W + q] = val[k * W + q];
        if (c == i) diag[i] = val[k * W];
    }
}

// Step k0 of the elimination, one block per kTile columns: D = A_kk^-1 (formed by every block for
// itself), the pivot rows R = D A_k,: (R_kk = D) and a copy C of the pivot columns.  Pivots up to `null`
// times their diagonal count as zero; *small is set where one above that is at most `low` times it.
template <bool CPLX>
__global__ void __launch_bounds__(256) k_gj_panel(int ld, int k0, double null, double low, const double* __restrict__ A,
                                                  const double* __restrict__ diag, double* __restrict__ R,
                                                  double* __restrict__ C, int* __restrict__ small) {
    constexpr int W = CPLX ? 2 : 1;
    __shared__ double M[W][kNb][kNb + 1];
    __shared__ double T[W][kNb][kTile + 4];
    __shared__ double rowp[2][W][kNb], colp[2][W][kNb];
    const int t = threadIdx.x, j0 = blockIdx.x * kTile;
    for (int e = t; e < kNb * kTile; e += 256) {
        const int i = e / kTile, j = e % kTile;
        for (int q = 0; q < W; q++) T[q][i][j] = A[(size_t(k0 + i) * ld + j0 + j) * W + q];
    }
    for (int e = t; e < kTile * kNb; e += 256) {
        const int i = e / kNb, j = e % kNb;
        for (int q = 0; q < W; q++) C[(size_t(j0 + i) * kNb + j) * W + q] = A[(size_t(j0 + i) * ld + k0 + j) * W + q];
    }
    // Gauss-Jordan on the diagonal block, elements (ri + 8 q, cj) in registers; the pivot row and
    // column go through LDS, two buffers in turn so that one barrier per pivot is enough
    const int cj = t % kNb, ri = t / kNb;
    double v[W][kNb / 8];
#pragma unroll
    for (int q = 0; q < kNb / 8; q++)
        for (int w = 0; w < W; w++) v[w][q] = A[(size_t(k0 + ri + 8 * q) * ld + k0 + cj) * W + w];
#pragma unroll
    for (int pq = 0; pq < kNb / 8; pq++)
        for (int pr = 0; pr < 8; pr++) {
            const int p = 8 * pq + pr, buf = p & 1;
            for (int w = 0; w < W; w++) {
                if (ri == pr) rowp[buf][w][cj] = v[w][pq];
                if (cj == p)
#pragma unroll
                    for (int q = 0; q < kNb / 8; q++) colp[buf][w][ri + 8 * q] = v[w][q];
            }
            __syncthreads();
            const double piv = rowp[buf][0][p], d = fabs(diag[k0 + p]);
            // A pivot that counts as zero: the unknown is left out (its row and column of the inverse are
            // zero), which solves every consistent system of a singular operator.  A clearly negative
            // one (an indefinite operator): a tiny pivot, as the host's Cholesky takes.
            const double ip = piv > null * d ? 1.0 / piv : piv >= -null * d ? 0.0 : 1.0 / fmax(1e-300, d * 1e-14 + 1e-300);
            if (blockIdx.x == 0 && t == 0 && piv > null * d && piv <= low * d) *small = 1;
            const double xr = rowp[buf][0][cj] * ip, xi = CPLX ? rowp[buf][W - 1][cj] * ip : 0.0;
#pragma unroll
            for (int q = 0; q < kNb / 8; q++) {
                const bool own = ri + 8 * q == p;
                const double lr = colp[buf][0][ri + 8 * q];
                if constexpr (CPLX) {
                    const double li = colp[buf][1][ri + 8 * q];
                    if (own) { v[0][q] = cj == p ? ip : xr; v[1][q] = cj == p ? 0.0 : xi; }
                    else if (cj == p) { v[0][q] = -lr * ip; v[1][q] = -li * ip; }
                    else { v[0][q] -= lr * xr - li * xi; v[1][q] -= lr * xi + li * xr; }
                } else {
                    v[0][q] = own ? (cj == p ? ip : xr) : cj == p ? -lr * ip : v[0][q] - lr * xr;
                }
            }
        }
#pragma unroll
    for (int q = 0; q < kNb / 8; q++)
        for (int w = 0; w < W; w++) M[w][ri + 8 * q][cj] = v[w][q];
    __syncthreads();
    // R tile = D T on the matrix cores: wavefront wid the 16 columns 16 wid .. of the tile
    const int lane = t & 63, wid = t >> 6, m = lane & 15, g = lane >> 4;
    d4 acc[2][W];
    for (int a = 0; a < 2; a++)
        for (int w = 0; w < W; w++) acc[a][w] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < kNb; kk += 4) {
        const double x0 = T[0][kk + g][16 * wid + m], x1 = CPLX ? T[W - 1][kk + g][16 * wid + m] : 0.0;
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const double c0 = M[0][16 * a + m][kk + g];
            acc[a][0] = mfma(c0, x0, acc[a][0]);
            if constexpr (CPLX) {
                const double c1 = M[1][16 * a + m][kk + g];
                acc[a][0] = mfma(-c1, x1, acc[a][0]);
                acc[a][1] = mfma(c0, x1, acc[a][1]);
                acc[a][1] = mfma(c1, x0, acc[a][1]);
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * a + g + 4 * r, j = j0 + 16 * wid + m;
            const bool own = j >= k0 && j < k0 + kNb;  // R_kk = D
            for (int w = 0; w < W; w++) R[(size_t(i) * ld + j) * W + w] = own ? M[w][i][j - k0] : acc[a][w][r];
        }
}

// A <- A - C R outside the pivot rows and columns; the pivot rows become R and the pivot columns
// -C D (their old value counts as zero, R_kk = D).  One kTile x kTile tile per block, a 32 x 32
// quarter per wavefront; bound by the matrix's own traffic (read and written once per step) above
// about 1,000 rows, by the two launches of a step below.
template <bool CPLX>
__global__ void __launch_bounds__(256) k_gj_update(int ld, int k0, double* __restrict__ A, const double* __restrict__ R,
                                                   const double* __restrict__ C) {
    constexpr int W = CPLX ? 2 : 1;
    __shared__ double sC[W][kTile][kNb + 1];
    __shared__ double sR[W][kNb][kTile + 4];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    const int i0 = blockIdx.y * kTile, j0 = blockIdx.x * kTile;
    for (int e = t; e < kTile * kNb; e += 256) {
        const int i = e / kNb, k = e % kNb;
        for (int q = 0; q < W; q++) sC[q][i][k] = -C[(size_t(i0 + i) * kNb + k) * W + q];
    }
    for (int e = t; e < kNb * kTile; e += 256) {
        const int k = e / kTile, j = e % kTile;
        for (int q = 0; q < W; q++) sR[q][k][j] = R[(size_t(k) * ld + j0 + j) * W + q];
    }
    __syncthreads();
    const int m = lane & 15, g = lane >> 4;
    const int wi = (wid >> 1) * 32, wj = (wid & 1) * 32;
    d4 acc[2][2][W];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + wi + 16 * a + g + 4 * r, j = j0 + wj + 16 * b + m;
                const bool pc = j >= k0 && j < k0 + kNb;
                for (int q = 0; q < W; q++) acc[a][b][q][r] = pc ? 0.0 : A[(size_t(i) * ld + j) * W + q];
            }
#pragma unroll
    for (int kk = 0; kk < kNb; kk += 4) {
        double c[2][W], x[2][W];
#pragma unroll
        for (int a = 0; a < 2; a++)
            for (int q = 0; q < W; q++) {
                c[a][q] = sC[q][wi + 16 * a + m][kk + g];
                x[a][q] = sR[q][kk + g][wj + 16 * a + m];
            }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                if constexpr (CPLX) {
                    acc[a][b][0] = mfma(c[a][0], x[b][0], acc[a][b][0]);
                    acc[a][b][0] = mfma(-c[a][1], x[b][1], acc[a][b][0]);
                    acc[a][b][1] = mfma(c[a][0], x[b][1], acc[a][b][1]);
                    acc[a][b][1] = mfma(c[a][1], x[b][0], acc[a][b][1]);
                } else {
                    acc[a][b][0] = mfma(c[a][0], x[b][0], acc[a][b][0]);
                }
            }
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + wi + 16 * a + g + 4 * r, j = j0 + wj + 16 * b + m;
                const bool pr = i >= k0 && i < k0 + kNb;
                for (int q = 0; q < W; q++)
                    A[(size_t(i) * ld + j) * W + q] =
                        pr ? R[(size_t(i - k0) * ld + j) * W + q] : acc[a][b][q][r];
            }
}

// x = Inv b: one wavefront per row, 16 bytes of the row per lane and load (two real columns or a
// complex one; ld is even, so rows stay aligned), kU loads in flight.
template <typename T, bool CPLX, bool DOTS>
__global__ void __launch_bounds__(256) k_dense_gemv(int n, int ld, const double* __restrict__ inv,
                                                    const T* __restrict__ b, T* __restrict__ x, const int* skip,
                                                    const double* __restrict__ r, const float* __restrict__ xold,
                                                    double* __restrict__ partials) {
    if (skip && *skip) return;
    const int row_ = blockIdx.x * 4 + int(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const bool in = row_ < n;  // uniform inside the wavefront
    if (!DOTS && !in) return;
    const int i = in ? row_ : n - 1;  // a wavefront past the end only takes part in the dots' reduction
    // the row's entries of r and xold, in flight with the row
    double rv[2] = {0.0, 0.0}, ov[2] = {0.0, 0.0};
    if (DOTS && in && lane == 0)
        for (int q = 0; q < (CPLX ? 2 : 1); q++) { rv[q] = r[(CPLX ? 2 : 1) * i + q]; ov[q] = double(xold[(CPLX ? 2 : 1) * i + q]); }
    constexpr int kU = 4;
    const double2* __restrict__ row = reinterpret_cast<const double2*>(inv + size_t(i) * ld * (CPLX ? 2 : 1));
    const int nv = CPLX ? n : (n + 1) / 2;  // 16-byte pieces; an odd n's last one ends in the padding
    double ar = 0.0, ai = 0.0;
    auto add = [&](const double2& m, int v) {
        const int j = 2 * v;
        const double b0 = double(b[j]);
        if constexpr (CPLX) {
            const double b1 = double(b[j + 1]);
            ar += m.x * b0 - m.y * b1;
            ai += m.x * b1 + m.y * b0;
        } else {
            ar += m.x * b0 + m.y * (j + 1 < n ? double(b[j + 1]) : 0.0);
        }
    };
    int v = lane;
    for (; v + (kU - 1) * 64 < nv; v += kU * 64) {
        double2 m[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) m[u] = row[v + 64 * u];
#pragma unroll
        for (int u = 0; u < kU; u++) add(m[u], v + 64 * u);
    }
    for (; v < nv; v += 64) add(row[v], v);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        ar += __shfl_xor(ar, off, 64);
        if constexpr (CPLX) ai += __shfl_xor(ai, off, 64);
    }
    if (lane == 0 && in) {
        if constexpr (CPLX) { x[2 * i] = T(ar); x[2 * i + 1] = T(ai); }
        else x[i] = T(ar);
    }
    if constexpr (DOTS) {
        double d[2] = {rv[0] * double(T(ar)) + rv[1] * double(T(ai)), rv[0] * ov[0] + rv[1] * ov[1]};
        partials_write<2>(d, partials);
    }
}

// X = Inv B for an n x MW row-major block: 16 rows per block of 1024 threads, 16 columns of B and
// one of the K splits per wavefront (4 column tiles x 4 splits at 64 columns, 1 x 16 at 16 and 8),
// on the FP64 matrix cores; the splits are added in order through LDS.  A lane reads the
// neighbours k, k + 1 of its row as 16 bytes and uses them in two products.  The one-thread-per-
// entry loop this replaces took 65 us at n = 280 and 97 us at n = 400 with 64 columns; this takes 14.4 us
// at n = 399 and 38 to 44 at n = 2,368 (45 MB; 148 blocks, so 108 of the 256 compute units are idle).
template <typename T, int MW>
__global__ void __launch_bounds__(1024) k_dense_block(int n, int ld, const double* __restrict__ inv,
                                                      const T* __restrict__ B, T* __restrict__ X, const int* skip) {
    if (skip && *skip) return;
    constexpr int CT = MW > 16 ? MW / 16 : 1;  // column tiles
    constexpr int KS = 16 / CT;                // splits of the inner dimension
    __shared__ double part[16][16][17];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int ct = wid % CT, ks = wid / CT;
    const int i0 = blockIdx.x * 16, j = ct * 16 + m;
    const int steps = ld / 8, per = (steps + KS - 1) / KS;
    const int s1 = min(steps, (ks + 1) * per);
    const double2* __restrict__ row = reinterpret_cast<const double2*>(inv + size_t(i0 + m) * ld);
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    // kU steps of 8 rows of B in flight; the last steps may reach past n (the padding of Inv's rows
    // is zero there, B is not read)
    constexpr int kU = 8;
    const T* __restrict__ Bj = B + (j < MW ? j : 0);
    int s = ks * per;
    for (; s + kU <= s1 && 8 * (s + kU) <= n; s += kU) {
        double2 a[kU];
        T b0[kU], b1[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int k = 8 * (s + u) + 2 * g;
            a[u] = row[k / 2];
            b0[u] = Bj[size_t(k) * MW];
            b1[u] = Bj[size_t(k + 1) * MW];
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            acc = mfma(a[u].x, double(b0[u]), acc);
            acc = mfma(a[u].y, double(b1[u]), acc);
        }
    }
    for (; s < s1; s++) {
        const int k = 8 * s + 2 * g;
        const double2 a = row[k / 2];
        acc = mfma(a.x, k < n ? double(Bj[size_t(k) * MW]) : 0.0, acc);
        acc = mfma(a.y, k + 1 < n ? double(Bj[size_t(k + 1) * MW]) : 0.0, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) part[wid][g + 4 * r][m] = acc[r];
    __syncthreads();
    const int oi = int(threadIdx.x) / MW, oj = int(threadIdx.x) % MW;
    if (oi < 16 && i0 + oi < n) {
        double v = 0.0;
        for (int q = 0; q < KS; q++) v += part[q * CT + oj / 16][oi][oj % 16];
        X[size_t(i0 + oi) * MW + oj] = T(v);
    }
}

}  // namespace

DenseInverse::DenseInverse(mk_ctx* c, bool cplx_, int n_, const int64_t* ptr, const int* col, const double* val,
                           bool fp32_null)
    : n(n_), ld((n_ + kTile - 1) / kTile * kTile), cplx(cplx_) {
    const size_t w = cplx ? 2 : 1, nz = size_t(ptr[n]);
    DevBuf<int64_t> dp;
    DevBuf<int> dc;
    DevBuf<double> dv, diag(static_cast<size_t>(ld)), R(size_t(kNb) * ld * w), C(size_t(kNb) * ld * w);
    dp.upload(ptr, size_t(n) + 1, c->stream);
    dc.upload(col, std::max<size_t>(nz, 1), c->stream);
    dv.upload(val, std::max<size_t>(nz, 1) * w, c->stream);
    inv.alloc(size_t(ld) * ld * w);
    const unsigned nt = unsigned(ld / kTile);
    // A pivot is its diagonal less squares that sum to at most it: n eps of it is rounding (measured 0.05
    // to 0.2 n eps on singular grids of 240 to 2,352 unknowns); a Galerkin operator's entries carry the
    // rounding of their own sums of tens of products.
    const double low = double(n) * 0x1p-23, null = fp32_null ? low : 32.0 * double(n) * 0x1p-52;
    DevBuf<int> small(1);
    MK_HIP(hipMemsetAsync(small.p, 0, sizeof(int), c->stream));
    auto run = [&](auto cp) {
        constexpr bool CP = decltype(cp)::value;
        hipLaunchKernelGGL((k_dense_fill<CP>), dim3(unsigned(ld)), dim3(256), 0, c->stream, n, ld,
                           (const int64_t*)dp.p, (const int*)dc.p, (const double*)dv.p, inv.p, diag.p);
        for (int k0 = 0; k0 < n; k0 += kNb) {
            hipLaunchKernelGGL((k_gj_panel<CP>), dim3(nt), dim3(256), 0, c->stream, ld, k0, null, low, (const double*)inv.p,
                               (const double*)diag.p, R.p, C.p, small.p);
            hipLaunchKernelGGL((k_gj_update<CP>), dim3(nt, nt), dim3(256), 0, c->stream, ld, k0, inv.p,
                               (const double*)R.p, (const double*)C.p);
        }
    };
    if (cplx) run(std::true_type{});
    else run(std::false_type{});
    MK_HIP(hipGetLastError());
    MK_HIP(hipMemcpyAsync(c->pin, small.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    MK_HIP(hipStreamSynchronize(c->stream));  // the temporaries are freed on return
    near_null = *static_cast<const int*>(c->pin) != 0;
}

template <typename T>
unsigned DenseInverse::apply(mk_ctx* c, const T* b, T* x, const int* skip, const double* r, const float* xold,
                             double* partials) const {
    const unsigned g = unsigned((n + 3) / 4);
#define MK_GEMV(CP, DOTS)                                                                                              \
    hipLaunchKernelGGL((k_dense_gemv<T, CP, DOTS>), dim3(g), dim3(256), 0, c->stream, n, ld, (const double*)inv.p, b, \
                       x, skip, r, xold, partials)
    constexpr bool dots = std::is_same<T, float>::value;  // only the FP32 V-cycle is asked for them
    MK_CHECK(dots || !r, MK_ERR_UNSUPPORTED, "dense product: dots in FP32 only");
    if (cplx) { if (r) MK_GEMV(true, dots); else MK_GEMV(true, false); }
    else { if (r) MK_GEMV(false, dots); else MK_GEMV(false, false); }
#undef MK_GEMV
    return g;
}
template unsigned DenseInverse::apply<float>(mk_ctx*, const float*, float*, const int*, const double*, const float*,
                                             double*) const;
template unsigned DenseInverse::apply<double>(mk_ctx*, const double*, double*, const int*, const double*, const float*,
                                              double*) const;

template <typename T>
void DenseInverse::apply_block(mk_ctx* c, int mw, const T* B, T* X, const int* skip) const {
    MK_CHECK(!cplx, MK_ERR_UNSUPPORTED, "dense block product: real inverses only");
    const dim3 g(unsigned(ld / 16));
#define MK_DENSE_BLOCK(MW)                                                                                         \
    hipLaunchKernelGGL((k_dense_block<T, MW>), g, dim3(1024), 0, c->stream, n, ld, (const double*)inv.p, B, X, skip)
    switch (mw) {
        case 8: MK_DENSE_BLOCK(8); break;
        case 16: MK_DENSE_BLOCK(16); break;
        case 32: MK_DENSE_BLOCK(32); break;
        case 64: MK_DENSE_BLOCK(64); break;
        default: throw Error(MK_ERR_ARG, "dense block product: block width must be 8, 16, 32 or 64");
    }
#undef MK_DENSE_BLOCK
}
template void DenseInverse::apply_block<float>(mk_ctx*, int, const float*, float*, const int*) const;
template void DenseInverse::apply_block<double>(mk_ctx*, int, const double*, double*, const int*) const;

}  // namespace mk
