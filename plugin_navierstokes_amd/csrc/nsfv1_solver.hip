// nsfv1_solver.hip -- device linear algebra for the Newton loop around the
// FV1 assembly: Dirichlet rows, CSR SpMV with the (FP32 or FP64) Jacobian on
// FP64 vectors, point-block Jacobi (one (dim+1)x(dim+1) block per node), and
// the BLAS-1 kernels of restarted GMRES.  All reductions use a fixed
// decomposition and order, so results are bitwise reproducible.
//
// The reference delegates this to ugcore (DirichletBoundary, NewtonSolver,
// linear solvers), which is not part of the plugin; these kernels provide the
// same service for the device-resident Jacobian and defect.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nsfv1_device.hpp"
#include "nsfv1_solver.hpp"

namespace nsfv1 {

// ---------------------------------------------------------------------
// Dirichlet rows: J row -> identity, d = u - g (ugcore DirichletBoundary
// row treatment, restated)
// ---------------------------------------------------------------------
template <typename JT>
__global__ void dirichlet_rows(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colidx,
                               const int64_t* __restrict__ rows, int64_t nrows, JT* __restrict__ J,
                               double* __restrict__ d, const double* __restrict__ u, const double* __restrict__ g)
{
    const int64_t r = (int64_t)blockIdx.x;
    if (r >= nrows) return;
    const int64_t row = rows[r];
    if (J)
        for (int64_t k = rowptr[row] + threadIdx.x; k < rowptr[row + 1]; k += blockDim.x)
            J[k] = colidx[k] == row ? JT(1) : JT(0);
    if (threadIdx.x == 0 && d) d[row] = u[row] - (g ? g[r] : 0.0);
}

// ---------------------------------------------------------------------
// y = A x, 16 lanes per row, fixed-order shuffle reduction
// ---------------------------------------------------------------------
template <typename JT>
__global__ void __launch_bounds__(256)
spmv_csr(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colidx, const JT* __restrict__ A,
         const double* __restrict__ x, double* __restrict__ y, int64_t n)
{
    const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    const int sub = threadIdx.x & 15;
    double s = 0.0;
    if (row < n) {
        const int64_t a = rowptr[row], b = rowptr[row + 1];
        for (int64_t k = a + sub; k < b; k += 16) s += (double)A[k] * x[colidx[k]];
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
    if (row < n && sub == 0) y[row] = s;
}

// ---------------------------------------------------------------------
// point-block Jacobi: invert the (nc x nc) diagonal block of every node
// (Gauss-Jordan with partial pivoting in FP64)
// ---------------------------------------------------------------------
template <typename JT, int NC>
__global__ void block_jacobi_setup(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colidx,
                                   const JT* __restrict__ A, int64_t nv, double* __restrict__ Binv,
                                   int* __restrict__ err)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    double M[NC][2 * NC];
    const int64_t r0 = rowptr[v * NC];
    const int deg = (int)((rowptr[v * NC + 1] - r0) / NC);
    // slot of the diagonal block in the row
    int lo = 0, hi = deg - 1, j = 0;
    const int32_t key = (int32_t)(v * NC);
    while (lo <= hi) {
        const int mid = (lo + hi) >> 1;
        const int32_t c = colidx[r0 + (int64_t)mid * NC];
        if (c == key) { j = mid; break; }
        if (c < key) lo = mid + 1; else hi = mid - 1;
    }
#pragma unroll
    for (int a = 0; a < NC; ++a) {
        const int64_t ra = rowptr[v * NC + a] + (int64_t)j * NC;
#pragma unroll
        for (int b = 0; b < NC; ++b) {
            M[a][b] = (double)A[ra + b];
            M[a][NC + b] = a == b ? 1.0 : 0.0;
        }
    }
    bool ok = true;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        int p = c;
        double best = fabs(M[c][c]);
#pragma unroll
        for (int r = c + 1; r < NC; ++r)
            if (fabs(M[r][c]) > best) { best = fabs(M[r][c]); p = r; }
        if (best == 0.0) { ok = false; break; }
        // swap rows c and p with compile-time indices only, so that M
        // stays in registers
#pragma unroll
        for (int r = c + 1; r < NC; ++r)
            if (r == p)
#pragma unroll
                for (int k = 0; k < 2 * NC; ++k) { const double t = M[c][k]; M[c][k] = M[r][k]; M[r][k] = t; }
        const double ip = 1.0 / M[c][c];
#pragma unroll
        for (int k = 0; k < 2 * NC; ++k) M[c][k] *= ip;
#pragma unroll
        for (int r = 0; r < NC; ++r)
            if (r != c) {
                const double f = M[r][c];
#pragma unroll
                for (int k = 0; k < 2 * NC; ++k) M[r][k] -= f * M[c][k];
            }
    }
#pragma unroll
    for (int a = 0; a < NC; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b) Binv[(v * NC + a) * NC + b] = ok ? M[a][NC + b] : (a == b ? 1.0 : 0.0);
    if (!ok) kernel_error(err, KERR_SINGULAR_BLOCK);
}

template <int NC>
__global__ void block_jacobi_apply(const double* __restrict__ Binv, const double* __restrict__ x,
                                   double* __restrict__ y, int64_t nv)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    double xv[NC];
#pragma unroll
    for (int a = 0; a < NC; ++a) xv[a] = x[v * NC + a];
#pragma unroll
    for (int a = 0; a < NC; ++a) {
        double s = 0;
#pragma unroll
        for (int b = 0; b < NC; ++b) s += Binv[(v * NC + a) * NC + b] * xv[b];
        y[v * NC + a] = s;
    }
}

// ---------------------------------------------------------------------
// BLAS-1 with deterministic two-stage reductions
// ---------------------------------------------------------------------
// Block sums of K values per thread, in a fixed order: the sum of value i ends
// in thread i.  Butterflies inside each wave, then the four waves in turn.
template <int K>
__device__ inline double block_sums(double (&v)[K], double (&sh)[4][K])
{
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < K; ++i) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_xor(v[i], o, 64);
        if (l == 0) sh[w][i] = v[i];
    }
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x < K)
        for (int q = 0; q < 4; ++q) t += sh[q][threadIdx.x];
    __syncthreads();
    return t;
}

// Orthogonalisation of w against V_0 .. V_{k-1} (classical Gram-Schmidt, twice).
// A workgroup holds 256 E entries of w in registers and walks the basis
// GS_VECS vectors at a time:
//   AXPY: w -= sum_i h_i V_i (w written), in ascending i;
//   DOT:  partial[i][block] = sum over the block of V_i . w (the updated w);
//   NORM: partial[0][block] = sum over the block of w^2.
// The update of one pass and the projections of the next share one launch, which
// reads its block's share of V twice; long vectors hold it in registers instead
// (gs_hold), since the share outlives the L2 only in part.  HBM bound: 2.3 M
// unknowns, mean k = 10.5: projections 48 us (4.4 TB/s), update and projections
// 84 us, update and norm 48 us; 3 launches of 180 us where dot and update in
// launches of their own took 261 us.
constexpr int GS_VECS = 8;

template <int E, bool AXPY, bool DOT, bool NORM, bool FULL>
__device__ __forceinline__ void gs_block(const double* __restrict__ V, int64_t ld, int k, const double* __restrict__ h,
                                         double* __restrict__ w, int64_t t0, int64_t n, double* __restrict__ part,
                                         double (&sh)[4][GS_VECS])
{
    // FULL: every entry of the block exists, so loads carry no mask
    const auto in = [&](int e) { return FULL || t0 + 256 * e < n; };
    double x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = in(e) ? w[t0 + 256 * e] : 0.0;
    if constexpr (AXPY) {
        int i = 0;
        for (; i + 2 <= k; i += 2) {
            const double h0 = h[i], h1 = h[i + 1];
            const double* v = V + i * ld + t0;
            double a[E], b[E];
#pragma unroll
            for (int e = 0; e < E; ++e) a[e] = in(e) ? v[256 * e] : 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) b[e] = in(e) ? v[ld + 256 * e] : 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = (x[e] - h0 * a[e]) - h1 * b[e];
        }
        if (i < k) {
            const double h0 = h[i];
            const double* v = V + i * ld + t0;
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] -= h0 * (in(e) ? v[256 * e] : 0.0);
        }
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (in(e)) w[t0 + 256 * e] = x[e];
    }
    if constexpr (DOT) {
        for (int i0 = 0; i0 < k; i0 += GS_VECS) {
            double acc[GS_VECS];
#pragma unroll
            for (int q = 0; q < GS_VECS; ++q) {
                acc[q] = 0.0;
                if (i0 + q < k) {
                    const double* v = V + (i0 + q) * ld + t0;
                    double a[E];
#pragma unroll
                    for (int e = 0; e < E; ++e) a[e] = in(e) ? v[256 * e] : 0.0;
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[q] += a[e] * x[e];
                }
            }
            const double s = block_sums(acc, sh);
            if (threadIdx.x < GS_VECS && i0 + (int)threadIdx.x < k) part[(int64_t)(i0 + threadIdx.x) * gridDim.x] = s;
        }
    }
    if constexpr (NORM) {
        double acc[GS_VECS] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int e = 0; e < E; ++e) acc[0] += x[e] * x[e];
        const double s = block_sums(acc, sh);
        if (threadIdx.x == 0) part[0] = s;
    }
}

template <int E, bool AXPY, bool DOT, bool NORM>
__global__ void __launch_bounds__(256)
gs_pass(const double* __restrict__ V, int64_t ld, int k, const double* __restrict__ h, double* __restrict__ w,
        int64_t n, double* __restrict__ partial)
{
    __shared__ double sh[4][GS_VECS];
    const int64_t b0 = (int64_t)blockIdx.x * (256 * E), t0 = b0 + threadIdx.x;
    double* part = partial + blockIdx.x;
    if (b0 + 256 * E <= n) gs_block<E, AXPY, DOT, NORM, true>(V, ld, k, h, w, t0, n, part, sh);
    else gs_block<E, AXPY, DOT, NORM, false>(V, ld, k, h, w, t0, n, part, sh);
}

// The update and the next projections of up to GS_HOLD vectors, KH of them (k
// rounded up to four, the surplus loads repeat the last vector) held in
// registers between the two: the basis streams once where gs_pass reads it
// twice (a block's share is 344 KB at k = 10).
// 2.3 M unknowns, k = 1 .. 20: 84 -> 52 us on average; 93 us at k = 17 .. 20 (4.3 TB/s).
// All three launches, 2.3 M unknowns: 276 us at k = 24 (4.8 TB/s), 381 us at k = 25,
// 451 at 30, 859 at 60 (3.6 to 3.9 TB/s): from 25 on, and below 2^20 unknowns
// (k = 8: 62 us just below, 49 us from there on), the basis is read twice.
constexpr int GS_HOLD = 24;

template <int E, int KH, bool FULL>
__device__ __forceinline__ void gs_hold_block(const double* __restrict__ V, int64_t ld, int k, const double* __restrict__ h,
                                              double* __restrict__ w, int64_t t0, int64_t n, double* __restrict__ part,
                                              double (&sh)[4][GS_VECS])
{
    const auto in = [&](int e) { return FULL || t0 + 256 * e < n; };
    double x[E], a[KH][E];
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = in(e) ? w[t0 + 256 * e] : 0.0;
#pragma unroll
    for (int i = 0; i < KH; ++i) {
        const double* v = V + (i < k ? i : k - 1) * ld + t0;
#pragma unroll
        for (int e = 0; e < E; ++e) a[i][e] = in(e) ? v[256 * e] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < KH; ++i) {
        if (i < k) {
            const double hi = h[i];
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] -= hi * a[i][e];
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (in(e)) w[t0 + 256 * e] = x[e];
#pragma unroll
    for (int i0 = 0; i0 < KH; i0 += GS_VECS) {
        double acc[GS_VECS];
#pragma unroll
        for (int q = 0; q < GS_VECS; ++q) {
            acc[q] = 0.0;
            if (i0 + q < KH)
#pragma unroll
                for (int e = 0; e < E; ++e) acc[q] += a[i0 + q < KH ? i0 + q : 0][e] * x[e];
        }
        const double s = block_sums(acc, sh);
        if (threadIdx.x < GS_VECS && i0 + (int)threadIdx.x < k) part[(int64_t)(i0 + threadIdx.x) * gridDim.x] = s;
    }
}

template <int E, int KH>
__global__ void __launch_bounds__(256)
gs_hold(const double* __restrict__ V, int64_t ld, int k, const double* __restrict__ h, double* __restrict__ w, int64_t n,
        double* __restrict__ partial)
{
    __shared__ double sh[4][GS_VECS];
    const int64_t b0 = (int64_t)blockIdx.x * (256 * E), t0 = b0 + threadIdx.x;
    double* part = partial + blockIdx.x;
    if (b0 + 256 * E <= n) gs_hold_block<E, KH, true>(V, ld, k, h, w, t0, n, part, sh);
    else gs_hold_block<E, KH, false>(V, ld, k, h, w, t0, n, part, sh);
}

// one workgroup per dot product: every thread sums a fixed strided subset
// of the partials, then the fixed-order block reduction (deterministic)
__global__ void __launch_bounds__(256)
multi_dot_final(const double* __restrict__ partial, int64_t nblk, double* __restrict__ out)
{
    __shared__ double sh[4][1];
    const int i = blockIdx.x;
    double s[1] = {0.0};
    for (int64_t b = threadIdx.x; b < nblk; b += blockDim.x) s[0] += partial[i * nblk + b];
    const double tot = block_sums(s, sh);
    if (threadIdx.x == 0) out[i] = tot;
}

// y = a x + b y; with b = 0, y is not read (it may hold anything, NaN
// bit patterns of a fresh allocation included)
__global__ void axpby(double a, const double* __restrict__ x, double b, double* __restrict__ y, int64_t n)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) y[t] = b == 0.0 ? a * x[t] : a * x[t] + b * y[t];
}

// ---------------------------------------------------------------------
// device-side GMRES of the capturable Newton step: the Hessenberg matrix,
// the Givens rotations and the back substitution stay on the device, so a
// fixed number of iterations runs without host synchronisation
// ---------------------------------------------------------------------
__global__ void fill_value(double* __restrict__ x, double v, int64_t n)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) x[t] = v;
}

// zeroes n 4-byte words (a kernel, not a memset node, so that a captured
// assembly replays it faithfully)
__global__ void zero_words(uint32_t* __restrict__ x, int64_t n)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) x[t] = 0u;
}

// beta = sqrt(||r||^2); the squared norm is also copied to res2 if given
__global__ void gm_beta(const double* __restrict__ n2, double* __restrict__ beta, double* __restrict__ res2)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        *beta = sqrt(*n2);
        if (res2) *res2 = *n2;
    }
}

// column j of the (m+1) x m Hessenberg matrix H (row-major) from the two
// classical Gram-Schmidt passes hd[0..j], hd[hs..hs+j] and ||w||^2 = hd[2 hs]
__global__ void gm_hcol(const double* __restrict__ hd, int hs, double* __restrict__ H, int m, int j)
{
    const int i = threadIdx.x;
    if (i <= j) H[i * m + j] = hd[i] + hd[hs + i];
    if (i == 0) H[(j + 1) * m + j] = sqrt(hd[2 * hs]);
}

// y = x / h, or 0 when h = 0 (a breakdown leaves a zero basis vector, whose
// Hessenberg column then vanishes)
__global__ void gm_scale(const double* __restrict__ x, const double* __restrict__ h, double* __restrict__ y, int64_t n)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double hv = *h;
    y[t] = hv > 0.0 ? x[t] / hv : 0.0;
}

// min ||beta e1 - H y|| over y (H overwritten by its rotated triangle):
// the Givens rotations of the host GMRES, then back substitution; a zero
// diagonal gives y_i = 0.  One thread (m <= GMRES_MAX_RESTART).
__global__ void gm_lsq(double* __restrict__ H, const double* __restrict__ beta, int m, double* __restrict__ y)
{
    __shared__ double g[GMRES_MAX_RESTART + 1], cs[GMRES_MAX_RESTART], sn[GMRES_MAX_RESTART];
    if (threadIdx.x != 0) return;
    for (int i = 0; i <= m; ++i) g[i] = 0.0;
    g[0] = *beta;
    for (int j = 0; j < m; ++j) {
        for (int i = 0; i < j; ++i) {
            const double t = cs[i] * H[i * m + j] + sn[i] * H[(i + 1) * m + j];
            H[(i + 1) * m + j] = -sn[i] * H[i * m + j] + cs[i] * H[(i + 1) * m + j];
            H[i * m + j] = t;
        }
        const double a = H[j * m + j], c = H[(j + 1) * m + j];
        const double r = hypot(a, c);
        cs[j] = r > 0 ? a / r : 1.0;
        sn[j] = r > 0 ? c / r : 0.0;
        H[j * m + j] = r;
        H[(j + 1) * m + j] = 0.0;
        g[j + 1] = -sn[j] * g[j];
        g[j] = cs[j] * g[j];
    }
    for (int i = m - 1; i >= 0; --i) {
        double t = g[i];
        for (int k = i + 1; k < m; ++k) t -= H[i * m + k] * y[k];
        y[i] = H[i * m + i] != 0.0 ? t / H[i * m + i] : 0.0;
    }
}

// x += sum_i c_i V_i
__global__ void multi_add(const double* __restrict__ V, int64_t ld, int k, const double* __restrict__ c,
                          double* __restrict__ x, int64_t n)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    double s = x[t];
    for (int i = 0; i < k; ++i) s += c[i] * V[i * ld + t];
    x[t] = s;
}


// ---------------------------------------------------------------------
// geometric multigrid pieces: residual, damped block-Jacobi update,
// node-level transfer operators, Dirichlet masking, state injection and
// the dense coarsest-level solve
// ---------------------------------------------------------------------

// Node-block products.  The pattern consists of (dim+1)x(dim+1) node
// blocks: node v has nb neighbours adj[off(v) + s] (off(v) = rowptr[v NC] /
// NC^2), and its NC rows all have nb NC entries, so entry (v a, s NC + c)
// sits at rowptr[v NC] + a nb NC + s NC + c.  A group of G lanes handles one
// node: lane j takes the slots s = j, j + G, ..., reads the neighbour index
// once and the NC x NC block as NC row segments (one 16-byte load per FP32
// row when NC = 4), and keeps NC FP64 partial sums.  The G partials are then
// combined by a reduce-scatter across the group (two exchange steps that
// halve the set of rows a lane carries, then a butterfly), in a fixed order.
// y = A x (RES = 0), y = b - A x with zeros in the rows of a mask (RES = 1),
// or one damped point-block Jacobi sweep y = x + omega Binv (b - A x) (RES = 2; y must not alias x).
template <typename JT, int NC>
__device__ __forceinline__ void block_row(const JT* __restrict__ p, double (&q)[NC])
{
#pragma unroll
    for (int c = 0; c < NC; ++c) q[c] = (double)p[c];
}
template <>
__device__ __forceinline__ void block_row<float, 4>(const float* __restrict__ p, double (&q)[4])
{
    const float4 t = *(const float4*)p;
    q[0] = t.x, q[1] = t.y, q[2] = t.z, q[3] = t.w;
}
template <>
__device__ __forceinline__ void block_row<double, 4>(const double* __restrict__ p, double (&q)[4])
{
    const double2 t0 = *(const double2*)p, t1 = *(const double2*)(p + 2);
    q[0] = t0.x, q[1] = t0.y, q[2] = t1.x, q[3] = t1.y;
}

template <typename JT, int NC, int G, int RES>
__global__ void __launch_bounds__(256)
nodeblock_mv(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ adj, const JT* __restrict__ A,
             const double* __restrict__ x, const double* __restrict__ b, double* __restrict__ y, int64_t nv,
             const double* __restrict__ Binv, double omega, const uint8_t* __restrict__ mask)
{
    static_assert(NC == 3 || NC == 4, "node blocks of 3 or 4 unknowns");
    static_assert(G >= 4 && G <= 64 && (G & (G - 1)) == 0, "group size");
    const int64_t v = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / G;
    const int sub = threadIdx.x & (G - 1);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (v < nv) {
        const int64_t base = rowptr[v * NC];
        const int nb = (int)((rowptr[v * NC + 1] - base) / NC);
        const int32_t* ad = adj + base / (NC * NC);
        const JT* Av = A + base;
#pragma unroll 2
        for (int sl = sub; sl < nb; sl += G) {
            const int64_t col = ad[sl];
            double xv[NC];
            if constexpr (NC == 4) {
                const double2 x0 = *(const double2*)(x + col * 4), x1 = *(const double2*)(x + col * 4 + 2);
                xv[0] = x0.x, xv[1] = x0.y, xv[2] = x1.x, xv[3] = x1.y;
            } else {
#pragma unroll
                for (int c = 0; c < NC; ++c) xv[c] = x[col * NC + c];
            }
#pragma unroll
            for (int a = 0; a < NC; ++a) {
                double q[NC];
                block_row<JT, NC>(Av + (int64_t)a * nb * NC + sl * NC, q);
                double t = acc[a];
#pragma unroll
                for (int c = 0; c < NC; ++c) t += q[c] * xv[c];
                acc[a] = t;
            }
        }
    }
    // reduce-scatter over the G lanes of the group: after the first step a
    // lane carries rows {0,1} or {2,3}, after the second one row
    const bool h1 = sub & (G / 2), h2 = sub & (G / 4);
    double w0, w1;
    {
        const double s0 = h1 ? acc[0] : acc[2], s1 = h1 ? acc[1] : acc[3];
        const double r0 = __shfl_xor(s0, G / 2, G), r1 = __shfl_xor(s1, G / 2, G);
        w0 = (h1 ? acc[2] : acc[0]) + r0;
        w1 = (h1 ? acc[3] : acc[1]) + r1;
    }
    double z = (h2 ? w1 : w0) + __shfl_xor(h2 ? w0 : w1, G / 4, G);
#pragma unroll
    for (int o = G / 8; o > 0; o >>= 1) z += __shfl_xor(z, o, G);
    const int a = (h1 ? 2 : 0) + (h2 ? 1 : 0);
    if constexpr (RES == 2) {
        // row c's sum sits on lane (c >> 1) G/2 + (c & 1) G/4 of the group
        double rr[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) rr[c] = __shfl(z, (c >> 1) * (G / 2) + (c & 1) * (G / 4), G);
        if (v < nv && (sub & (G / 4 - 1)) == 0 && a < NC) {
#pragma unroll
            for (int c = 0; c < NC; ++c) rr[c] = b[v * NC + c] - rr[c];
            const int64_t row = v * NC + a;
            double t = 0;
#pragma unroll
            for (int c = 0; c < NC; ++c) t += Binv[row * NC + c] * rr[c];
            y[row] = x[row] + omega * t;
        }
    } else if (v < nv && (sub & (G / 4 - 1)) == 0 && a < NC) {
        const int64_t row = v * NC + a;
        y[row] = RES ? (mask && mask[row] ? 0.0 : b[row] - z) : z;
    }
}

template <typename JT>
__global__ void __launch_bounds__(256)
residual_csr(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colidx, const JT* __restrict__ A,
             const double* __restrict__ x, const double* __restrict__ b, double* __restrict__ r, int64_t n,
             const uint8_t* __restrict__ mask)
{
    const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    const int sub = threadIdx.x & 15;
    double s = 0.0;
    if (row < n) {
        const int64_t a = rowptr[row], e = rowptr[row + 1];
        for (int64_t k = a + sub; k < e; k += 16) s += (double)A[k] * x[colidx[k]];
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
    if (row < n && sub == 0) r[row] = mask && mask[row] ? 0.0 : b[row] - s;
}

// x = (first ? 0 : x) + omega * Binv r, per node block
template <int NC>
__global__ void bj_update(const double* __restrict__ Binv, const double* __restrict__ r, double* __restrict__ x,
                          double omega, int first, int64_t nv)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    double rv[NC];
#pragma unroll
    for (int a = 0; a < NC; ++a) rv[a] = r[v * NC + a];
#pragma unroll
    for (int a = 0; a < NC; ++a) {
        double s = 0;
#pragma unroll
        for (int b = 0; b < NC; ++b) s += Binv[(v * NC + a) * NC + b] * rv[b];
        x[v * NC + a] = (first ? 0.0 : x[v * NC + a]) + omega * s;
    }
}

// y[row, c] = base[row, c] + sum_k w_k x[col_k, c] for every component c < nc
// (base may be null: 0); where the mask is set the sum is dropped
__global__ void node_transfer(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colidx,
                              const double* __restrict__ w, const double* __restrict__ x, const double* base,
                              const uint8_t* __restrict__ mask, double* y, int64_t nrows, int nc)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nrows * nc) return;
    const int64_t row = t / nc;
    const int c = (int)(t - row * nc);
    double s = 0.0;
    const int64_t a = rowptr[row], b = rowptr[row + 1];
    // unrolled so that several index -> value load chains are in flight
#pragma unroll 4
    for (int64_t k = a; k < b; ++k) s += w[k] * x[(int64_t)colidx[k] * nc + c];
    if (mask && mask[t]) s = 0.0;
    y[t] = base ? base[t] + s : s;
}

// coarse state: uc[w, c] = uf[inj[w], c]
__global__ void inject_state(const int64_t* __restrict__ inj, const double* __restrict__ uf, double* __restrict__ uc,
                             int64_t nvc, int nc)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nvc * nc) return;
    const int64_t w = t / nc;
    const int c = (int)(t - w * nc);
    uc[t] = uf[inj[w] * nc + c];
}

// y = A x with a dense row-major n x n matrix, one wavefront per row
__global__ void __launch_bounds__(256)
dense_matvec(const double* __restrict__ A, const double* __restrict__ x, double* __restrict__ y, int n)
{
    const int row = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int lane = threadIdx.x & 63;
    double s = 0.0;
    if (row < n)
        for (int k = lane; k < n; k += 64) s += A[(int64_t)row * n + k] * x[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (row < n && lane == 0) y[row] = s;
}

// ---------------------------------------------------------------------
// coarsest-level dense inverse: Gauss-Jordan in exchange form with partial
// pivoting and no row swaps.  The tableau y = M x starts as the coarse
// matrix; step k takes the unpivoted row p with the largest |M[p][k]| and
// exchanges y_p with x_k:
//   M'[p][k] = 1/a, M'[p][j] = -M[p][j]/a,
//   M'[i][k] = M[i][k]/a, M'[i][j] = M[i][j] - M'[i][k] M[p][j]   (i != p),
// a = M[p][k].  After n steps x_k = sum_j M[p_k][j] y_{p_j}, so
// inv[k][p_j] = M[p_k][j].  Ties of the pivot search go to the smaller row.
// A column that vanishes on every unpivoted row (a null mode of the coarse
// operator, e.g. the constant pressure of a domain with Dirichlet velocity
// everywhere) pins its unknown to zero in the coarse correction (a = 0 is
// replaced by 1/a := 0), instead of dividing by zero; a column with no
// finite entry left is reported.
//
// GJ_BLOCK steps form a panel.  Its columns, exchanged step by step, hold
// G = A A_pp^-1 in the end (A the panel's columns, A_pp its pivot rows; A_pp^-1
// itself in the pivot rows), so on the other columns the panel is one product
// M' = C - G M_p with M_p the pivot rows before the panel and C = M, or 0 in the
// pivot rows.  gj_step applies panel k to ping-pong tableaux, one wave per 16
// rows on the FP64 matrix cores; its first workgroup meanwhile brings the
// columns of panel k + 1 up to date with the same products and exchanges them,
// rows in registers, and leaves their G for the next launch.
//
// The bound is the dependent chain of the pivots (search, one barrier, one
// division, one row update), so it stays in one workgroup without a global
// access, with few waves (each instruction of the search costs every wave),
// and everything else runs beside it.  The search compares the upper 32 bits of
// the sizes: the pivot is the largest to a factor 1 + 2^-20.
// Measured: 16 pivots take 28 us of a launch's 36 us; n = 867: 2.1 ms (four
// pivots per launch, each workgroup repeating the search: 7.2 ms), n = 448:
// 0.8 ms (1.9 ms).  512 threads beat 256 (37.0 us a launch: the loads of the
// next panel's columns) and 1024 (51 us: the search).
// ---------------------------------------------------------------------
template <typename JT>
__global__ void __launch_bounds__(256)
gj_load(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ colidx, const JT* __restrict__ J, int n,
        double* __restrict__ M, int* __restrict__ done, int* __restrict__ err)
{
    const int r = blockIdx.x;
    double* row = M + (int64_t)r * n;
    for (int j = threadIdx.x; j < n; j += blockDim.x) row[j] = 0.0;
    __syncthreads();
    for (int64_t k = rowptr[r] + threadIdx.x; k < rowptr[r + 1]; k += blockDim.x) row[colidx[k]] = (double)J[k];
    if (threadIdx.x == 0) {
        done[r] = 0;
        if (r == 0) *err = 0;
    }
}

constexpr int GJ_BLOCK = 16;  // pivots of a panel
constexpr int GJ_TPB = 512;
typedef double f64x4 __attribute__((ext_vector_type(4)));

// what a panel leaves for its update
struct GJPanel {
    double* G;  // [n][GJ_BLOCK], 0 past the panel's last column
    int* flag;  // [n]: 1 for the rows pivoted in the panel
    int* piv;   // [GJ_BLOCK]: pivot rows, -1 past the last step
};

// pivot rows of the panel at columns j0 ..: B operands of the four products
// (lane l: row 4 s + (l >> 4), column l & 15)
__device__ __forceinline__ void gj_pivot_rows(const double* __restrict__ M, const GJPanel& G, int n, int j0, int lane,
                                              double (&P)[GJ_BLOCK / 4])
{
    const int j = j0 + (lane & 15) < n ? j0 + (lane & 15) : n - 1;
#pragma unroll
    for (int s = 0; s < GJ_BLOCK / 4; ++s) {
        const int r = G.piv[4 * s + (lane >> 4)];
        const double m = M[r > 0 ? r * n + j : j];
        P[s] = r >= 0 ? m : 0.0;
    }
}

// 16 x 16 tile at (r0, j0) of C - G M_p: lane l holds column l & 15, rows
// (l >> 4) + 4 i (the FP64 16x16x4 accumulator layout).  Loads are
// unconditional (indices clamped; what lies outside the tableau is not used),
// so that those of several tiles are in flight together.
struct GJTile {
    double c[4], g[GJ_BLOCK / 4];
    int flag[4];
};

__device__ __forceinline__ void gj_load_tile(const double* __restrict__ M, const GJPanel& G, int n, int r0, int j0,
                                             int lane, GJTile& T)
{
    const int cl = lane & 15, kq = lane >> 4;
    const int j = j0 + cl < n ? j0 + cl : n - 1, ra = r0 + cl < n ? r0 + cl : n - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = r0 + kq + 4 * i < n ? r0 + kq + 4 * i : n - 1;
        T.c[i] = M[r * n + j];
        T.flag[i] = G.flag[r];
    }
#pragma unroll
    for (int s = 0; s < GJ_BLOCK / 4; ++s) T.g[s] = G.G[ra * GJ_BLOCK + 4 * s + kq];
}

__device__ __forceinline__ f64x4 gj_tile(const GJTile& T, const double (&P)[GJ_BLOCK / 4])
{
    f64x4 acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = T.flag[i] ? 0.0 : T.c[i];
#pragma unroll
    for (int s = 0; s < GJ_BLOCK / 4; ++s) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-T.g[s], P[s], acc, 0, 0, 0);
    return acc;
}

template <int ROR>
__device__ __forceinline__ uint32_t row_max_step(uint32_t v)
{
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x120 + ROR, 0xf, 0xf, false);
    return v > o ? v : o;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    v = row_max_step<8>(v);
    v = row_max_step<4>(v);
    v = row_max_step<2>(v);
    v = row_max_step<1>(v);
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    const uint32_t ab = a > b ? a : b, cd = c > d ? c : d;
    return ab > cd ? ab : cd;
}

struct GJSlot {
    double row[GJ_BLOCK];
    uint32_t key;
    int r;
};

// The nb pivots of a panel, row t + GJ_TPB h in thread t, the panel's values in
// registers.  The registers rotate, pan[h][0] being the column of the current
// step: a step writes column x + 1 to register x and the step's own column to
// the last one, so every index is a compile-time constant.
template <int R>
__device__ __forceinline__ void gj_pivots(double (&pan)[R][GJ_BLOCK], int (&dn)[R], int (&in)[R],
                                          GJSlot (&slot)[2][GJ_TPB / 64], int (&sp)[GJ_BLOCK], int& bad, int n, int nb,
                                          int t, int lane, int wave)
{
    constexpr int B = GJ_BLOCK, W = GJ_TPB / 64;
    // sort keys: 0 for pivoted rows, NaN and rows past the end
    const auto sort_key = [](double v, int pivoted) {
        const double a = fabs(v);
        return (pivoted || a != a) ? 0u : (uint32_t)(__builtin_bit_cast(uint64_t, a) >> 32) + 1u;
    };
    uint32_t key[R], mx = 0;
#pragma unroll
    for (int h = 0; h < R; ++h) {
        key[h] = sort_key(pan[h][0], dn[h]);
        mx = key[h] > mx ? key[h] : mx;
    }
    mx = wave_max(mx);
#pragma unroll 1
    for (int q = 0; q < nb; ++q) {
        // the wave's smallest row of the largest key publishes its panel row
        GJSlot& sl = slot[q & 1][wave];
        bool open = true;
#pragma unroll
        for (int h = 0; h < R; ++h) {
            const uint64_t hit = __ballot(key[h] == mx);
            if (open && hit != 0) {
                open = false;
                if (lane == (int)__builtin_ctzll(hit)) {
#pragma unroll
                    for (int x = 0; x < B; ++x) sl.row[x] = pan[h][x];
                    sl.key = mx;
                    sl.r = t + GJ_TPB * h;
                }
            }
        }
        __syncthreads();
        // best of the waves (ties: the smaller row)
        const uint32_t ks = slot[q & 1][lane & (W - 1)].key;
        const int rs = slot[q & 1][lane & (W - 1)].r;
        int w = 0, p = __builtin_amdgcn_readlane(rs, 0);
        uint32_t best = (uint32_t)__builtin_amdgcn_readlane((int)ks, 0);
#pragma unroll
        for (int o = 1; o < W; ++o) {
            const uint32_t k2 = (uint32_t)__builtin_amdgcn_readlane((int)ks, o);
            const int p2 = __builtin_amdgcn_readlane(rs, o);
            if (k2 > best || (k2 == best && p2 < p)) {
                best = k2;
                p = p2;
                w = o;
            }
        }
        double pr[B];
#pragma unroll
        for (int x = 0; x < B; ++x) pr[x] = slot[q & 1][w].row[x];
        const double ia = pr[0] == 0.0 ? 0.0 : 1.0 / pr[0];
        if (t == 0) sp[q] = p;
        bad |= best == 0;
        // the next step's column first: its search runs beside the other columns
        double f[R];
        mx = 0;
#pragma unroll
        for (int h = 0; h < R; ++h) {
            f[h] = pan[h][0] * ia;
            pan[h][0] = fma(-f[h], pr[1], pan[h][1]);
            if (t + GJ_TPB * h == p) dn[h] = in[h] = 1;
            key[h] = sort_key(pan[h][0], dn[h]);
            mx = key[h] > mx ? key[h] : mx;
        }
        mx = wave_max(mx);
#pragma unroll
        for (int h = 0; h < R; ++h) {
#pragma unroll
            for (int x = 1; x + 1 < B; ++x) pan[h][x] = fma(-f[h], pr[x + 1], pan[h][x + 1]);
            pan[h][B - 1] = f[h];
        }
        if (((p >> 6) & (W - 1)) == wave)
#pragma unroll
            for (int h = 0; h < R; ++h)
                if (t + GJ_TPB * h == p) {  // the pivot row
#pragma unroll
                    for (int x = 0; x + 1 < B; ++x) pan[h][x] = -pr[x + 1] * ia;
                    pan[h][B - 1] = ia;
                }
    }
    // a short last panel: rotate on until column x sits in register x
#pragma unroll 1
    for (int q = nb; q < B; ++q) {
#pragma unroll
        for (int h = 0; h < R; ++h) {
            const double v = pan[h][0];
#pragma unroll
            for (int x = 0; x + 1 < B; ++x) pan[h][x] = pan[h][x + 1];
            pan[h][B - 1] = v;
        }
        if (t == 0) sp[q] = -1;
    }
}

// R rows of the panel per thread (n <= GJ_TPB R)
template <int R>
__global__ void __launch_bounds__(GJ_TPB)
gj_step(const double* __restrict__ Min, double* __restrict__ Mout, GJPanel cur, GJPanel nxt, int* __restrict__ done,
        int* __restrict__ piv, int* __restrict__ err, int n, int k0, int first)
{
    constexpr int B = GJ_BLOCK;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    if (blockIdx.x > 0) {
        // update: one 16 x 16 tile per wave
        const int tiles = (n + B - 1) / B;
        const int tile = ((int)blockIdx.x - 1) * (GJ_TPB / 64) + wave;
        const int j0 = (tile % tiles) * B, r0 = (tile / tiles) * B;
        if (r0 >= n) return;
        const int j = j0 + (lane & 15);
        f64x4 v;
        if (j0 == k0) {  // the panel's own columns: G
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = r0 + (lane >> 4) + 4 * i;
                v[i] = r < n ? cur.G[(int64_t)r * B + (lane & 15)] : 0.0;
            }
        } else {
            double P[B / 4];
            GJTile T;
            gj_load_tile(Min, cur, n, r0, j0, lane, T);
            gj_pivot_rows(Min, cur, n, j0, lane, P);
            v = gj_tile(T, P);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + (lane >> 4) + 4 * i;
            if (r < n && j < n) Mout[(int64_t)r * n + j] = v[i];
        }
        return;
    }

    // the next panel: columns [k1, k1 + nb)
    __shared__ double stage[GJ_TPB / 64][16][17];  // per wave: one tile, to hand its rows to lanes
    __shared__ GJSlot slot[2][GJ_TPB / 64];
    __shared__ int sp[B];
    const int k1 = first ? 0 : k0 + B;
    if (k1 >= n) return;
    const int nb = n - k1 < B ? n - k1 : B;
    double pan[R][B];
    int dn[R], in[R];
#pragma unroll
    for (int h = 0; h < R; ++h) {
        const int r = t + GJ_TPB * h;
        dn[h] = r < n ? done[r] : 1;
        in[h] = 0;
#pragma unroll
        for (int x = 0; x < B; ++x) pan[h][x] = 0.0;
    }
    double P[B / 4];
    if (!first) gj_pivot_rows(Min, cur, n, k1, lane, P);
#pragma unroll
    for (int h = 0; h < R; ++h) {
        f64x4 v[4];
        GJTile T[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) gj_load_tile(Min, cur, n, GJ_TPB * h + wave * 64 + q * 16, k1, lane, T[q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!first) {
                v[q] = gj_tile(T[q], P);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[q][i] = T[q].c[i];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int i = 0; i < 4; ++i) stage[wave][(lane >> 4) + 4 * i][lane & 15] = v[q][i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            // every lane reads (row lane & 15); the tile's lanes keep it
#pragma unroll
            for (int x = 0; x < B; ++x) {
                const double w = stage[wave][lane & 15][x];
                pan[h][x] = (lane >> 4) == q ? w : pan[h][x];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    int bad = 0;
    gj_pivots<R>(pan, dn, in, slot, sp, bad, n, nb, t, lane, wave);
    __syncthreads();
    if (t < B) {
        nxt.piv[t] = sp[t];
        if (t < nb) piv[k1 + t] = sp[t];
    }
    if (t == 0 && bad) *err = 1;
#pragma unroll
    for (int h = 0; h < R; ++h) {
        const int r = t + GJ_TPB * h;
        if (r >= n) continue;
        done[r] = dn[h];
        nxt.flag[r] = in[h];
#pragma unroll
        for (int x = 0; x < B; ++x) nxt.G[(int64_t)r * B + x] = x < nb ? pan[h][x] : 0.0;
    }
}

__global__ void gj_unpermute(const double* __restrict__ M, const int* __restrict__ piv, int n, double* __restrict__ inv)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * n) return;
    const int k = (int)(e / n), j = (int)(e - (int64_t)k * n);
    inv[(int64_t)k * n + piv[j]] = M[(int64_t)piv[k] * n + j];
}

// ---------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------
static inline int blocks_for(int64_t n, int t) { return (int)((n + t - 1) / t); }

hipError_t launch_dirichlet(int jprec, const int64_t* rowptr, const int32_t* colidx, const int64_t* rows,
                            int64_t nrows, void* J, double* d, const double* u, const double* g, hipStream_t s)
{
    if (nrows <= 0) return hipSuccess;
    if (jprec == 64)
        dirichlet_rows<double><<<(unsigned)nrows, 64, 0, s>>>(rowptr, colidx, rows, nrows, (double*)J, d, u, g);
    else
        dirichlet_rows<float><<<(unsigned)nrows, 64, 0, s>>>(rowptr, colidx, rows, nrows, (float*)J, d, u, g);
    return hipGetLastError();
}

// node-block launch: G lanes per node, the power of two (8, 16 or 32) that covers
// the mean number of neighbour blocks per node; 4 lanes for the 7 to 12 blocks of
// quadrilaterals (two or three blocks each: fewer lanes idle, two exchange steps
// less).  0.77 M nodes of 9 blocks, FP32 77 -> 65 us, FP64 150 us with either; 16 k
// nodes 3.8 -> 3.2 and 4.6 -> 3.7 us.  Triangles (7 blocks less the boundary's share,
// always below 7) keep 8: with 4 lanes 0.77 M nodes 47 us in FP32 as well, but
// 124 against 88 us in FP64, and 1 k nodes 3.0 against 2.7 us.
template <typename JT, int NC, int RES>
static void launch_nodeblock(const int64_t* rowptr, const int32_t* adj, const JT* A, const double* x, const double* b,
                             double* y, int64_t nv, int64_t nnz, const double* Binv, double omega,
                             const uint8_t* mask, hipStream_t s)
{
    const int64_t slots = nv > 0 ? nnz / ((int64_t)NC * NC * nv) : 0;
    if (NC == 3 && slots >= 7 && slots <= 12)
        nodeblock_mv<JT, NC, 4, RES><<<blocks_for(nv * 4, 256), 256, 0, s>>>(rowptr, adj, A, x, b, y, nv, Binv, omega, mask);
    else if (slots > 16)
        nodeblock_mv<JT, NC, 32, RES><<<blocks_for(nv * 32, 256), 256, 0, s>>>(rowptr, adj, A, x, b, y, nv, Binv, omega, mask);
    else if (slots > 8)
        nodeblock_mv<JT, NC, 16, RES><<<blocks_for(nv * 16, 256), 256, 0, s>>>(rowptr, adj, A, x, b, y, nv, Binv, omega, mask);
    else
        nodeblock_mv<JT, NC, 8, RES><<<blocks_for(nv * 8, 256), 256, 0, s>>>(rowptr, adj, A, x, b, y, nv, Binv, omega, mask);
}

// with 4 unknowns per node the node-block kernels take 16-byte vector loads
// of A and x
static bool nodeblock_ok(const int32_t* adj, int nc, const void* A, const double* x)
{
    return adj && (nc == 3 || (nc == 4 && (((uintptr_t)A | (uintptr_t)x) & 15) == 0));
}

template <int RES>
static void launch_mv(int jprec, const int64_t* rowptr, const int32_t* adj, int nc, const void* A, const double* x,
                      const double* b, double* y, int64_t n, int64_t nnz, hipStream_t s,
                      const double* Binv = nullptr, double omega = 0.0, const uint8_t* mask = nullptr)
{
    const int64_t nv = n / nc;
    if (nc == 4) {
        if (jprec == 64) launch_nodeblock<double, 4, RES>(rowptr, adj, (const double*)A, x, b, y, nv, nnz, Binv, omega, mask, s);
        else launch_nodeblock<float, 4, RES>(rowptr, adj, (const float*)A, x, b, y, nv, nnz, Binv, omega, mask, s);
    } else {
        if (jprec == 64) launch_nodeblock<double, 3, RES>(rowptr, adj, (const double*)A, x, b, y, nv, nnz, Binv, omega, mask, s);
        else launch_nodeblock<float, 3, RES>(rowptr, adj, (const float*)A, x, b, y, nv, nnz, Binv, omega, mask, s);
    }
}

hipError_t launch_spmv(int jprec, const int64_t* rowptr, const int32_t* colidx, const int32_t* adj, int nc,
                       const void* A, const double* x, double* y, int64_t n, int64_t nnz, hipStream_t s)
{
    if (nodeblock_ok(adj, nc, A, x)) {
        launch_mv<0>(jprec, rowptr, adj, nc, A, x, nullptr, y, n, nnz, s);
    } else {
        const int bl = blocks_for(n * 16, 256);
        if (jprec == 64) spmv_csr<double><<<bl, 256, 0, s>>>(rowptr, colidx, (const double*)A, x, y, n);
        else spmv_csr<float><<<bl, 256, 0, s>>>(rowptr, colidx, (const float*)A, x, y, n);
    }
    return hipGetLastError();
}

hipError_t launch_block_jacobi_setup(int jprec, int nc, const int64_t* rowptr, const int32_t* colidx, const void* A,
                                     int64_t nv, double* Binv, int* err, hipStream_t s)
{
    const int bl = blocks_for(nv, 128);
    if (nc == 3) {
        if (jprec == 64) block_jacobi_setup<double, 3><<<bl, 128, 0, s>>>(rowptr, colidx, (const double*)A, nv, Binv, err);
        else block_jacobi_setup<float, 3><<<bl, 128, 0, s>>>(rowptr, colidx, (const float*)A, nv, Binv, err);
    } else {
        if (jprec == 64) block_jacobi_setup<double, 4><<<bl, 128, 0, s>>>(rowptr, colidx, (const double*)A, nv, Binv, err);
        else block_jacobi_setup<float, 4><<<bl, 128, 0, s>>>(rowptr, colidx, (const float*)A, nv, Binv, err);
    }
    return hipGetLastError();
}

hipError_t launch_block_jacobi_apply(int nc, const double* Binv, const double* x, double* y, int64_t nv, hipStream_t s)
{
    const int bl = blocks_for(nv, 256);
    if (nc == 3) block_jacobi_apply<3><<<bl, 256, 0, s>>>(Binv, x, y, nv);
    else block_jacobi_apply<4><<<bl, 256, 0, s>>>(Binv, x, y, nv);
    return hipGetLastError();
}

// entries of w per thread: 16 fill the chip from 2^20 unknowns on (256
// workgroups) and amortise the block sums; below, 4 give more workgroups
static inline bool gs_wide(int64_t n) { return n >= (int64_t)1 << 20; }
static inline int64_t gs_blocks(int64_t n) { return (n + (gs_wide(n) ? 4096 : 1024) - 1) / (gs_wide(n) ? 4096 : 1024); }

// (the held basis takes blocks of 512 or 1024 entries)
int64_t red_partials(int64_t n)
{
    const int64_t nb = gs_wide(n) ? (n + 511) / 512 : gs_blocks(n);
    return 64 * (nb > 0 ? nb : 1);
}

template <bool AXPY, bool DOT, bool NORM>
static hipError_t launch_gs(const double* V, int64_t ld, int k, const double* h, double* w, int64_t n, double* partial,
                            double* out, hipStream_t s)
{
    if (n <= 0 || k < 0 || k > 64) return hipErrorInvalidValue;
    const int64_t nb = gs_blocks(n);
    if (gs_wide(n)) gs_pass<16, AXPY, DOT, NORM><<<(unsigned)nb, 256, 0, s>>>(V, ld, k, h, w, n, partial);
    else gs_pass<4, AXPY, DOT, NORM><<<(unsigned)nb, 256, 0, s>>>(V, ld, k, h, w, n, partial);
    const int nout = NORM ? 1 : k;
    if (nout > 0) multi_dot_final<<<nout, 256, 0, s>>>(partial, nb, out);
    return hipGetLastError();
}

hipError_t launch_norm2(const double* w, int64_t n, double* partial, double* out, hipStream_t s)
{
    return launch_gs<false, false, true>(nullptr, 0, 0, nullptr, const_cast<double*>(w), n, partial, out, s);
}

static hipError_t launch_gs_hold(const double* V, int64_t ld, int k, const double* h, double* w, int64_t n,
                                 double* partial, double* out, hipStream_t s)
{
    const int64_t nb = (n + (k <= 16 ? 1023 : 511)) / (k <= 16 ? 1024 : 512);
    const unsigned g = (unsigned)nb;
    switch ((k + 3) / 4) {
    case 1: gs_hold<4, 4><<<g, 256, 0, s>>>(V, ld, k, h, w, n, partial); break;
    case 2: gs_hold<4, 8><<<g, 256, 0, s>>>(V, ld, k, h, w, n, partial); break;
    case 3: gs_hold<4, 12><<<g, 256, 0, s>>>(V, ld, k, h, w, n, partial); break;
    case 4: gs_hold<4, 16><<<g, 256, 0, s>>>(V, ld, k, h, w, n, partial); break;
    case 5: gs_hold<2, 20><<<g, 256, 0, s>>>(V, ld, k, h, w, n, partial); break;
    case 6: gs_hold<2, 24><<<g, 256, 0, s>>>(V, ld, k, h, w, n, partial); break;
    default: return hipErrorInvalidValue;
    }
    multi_dot_final<<<k, 256, 0, s>>>(partial, nb, out);
    return hipGetLastError();
}

hipError_t launch_orthogonalise(const double* V, int64_t ld, int k, double* w, int64_t n, double* partial, double* h,
                                int hs, hipStream_t s)
{
    if (k < 1 || k > hs) return hipErrorInvalidValue;
    hipError_t e = launch_gs<false, true, false>(V, ld, k, nullptr, w, n, partial, h, s);
    if (e == hipSuccess)
        e = gs_wide(n) && k <= GS_HOLD ? launch_gs_hold(V, ld, k, h, w, n, partial, h + hs, s)
                                       : launch_gs<true, true, false>(V, ld, k, h, w, n, partial, h + hs, s);
    if (e == hipSuccess) e = launch_gs<true, false, true>(V, ld, k, h + hs, w, n, partial, h + 2 * hs, s);
    return e;
}

hipError_t launch_multi_add(const double* V, int64_t ld, int k, const double* c, double* x, int64_t n, hipStream_t s)
{
    multi_add<<<blocks_for(n, 256), 256, 0, s>>>(V, ld, k, c, x, n);
    return hipGetLastError();
}

hipError_t launch_axpby(double a, const double* x, double b, double* y, int64_t n, hipStream_t s)
{
    axpby<<<blocks_for(n, 256), 256, 0, s>>>(a, x, b, y, n);
    return hipGetLastError();
}

hipError_t launch_zero_words(void* x, int64_t nwords, hipStream_t s)
{
    if (nwords <= 0) return hipSuccess;
    zero_words<<<blocks_for(nwords, 256), 256, 0, s>>>(static_cast<uint32_t*>(x), nwords);
    return hipGetLastError();
}

hipError_t launch_fill(double* x, double v, int64_t n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    fill_value<<<blocks_for(n, 256), 256, 0, s>>>(x, v, n);
    return hipGetLastError();
}

hipError_t launch_gm_beta(const double* n2, double* beta, double* res2, hipStream_t s)
{
    gm_beta<<<1, 64, 0, s>>>(n2, beta, res2);
    return hipGetLastError();
}

hipError_t launch_gm_hcol(const double* hd, int hs, double* H, int m, int j, hipStream_t s)
{
    if (j < 0 || j >= m || m > GMRES_MAX_RESTART || hs < m) return hipErrorInvalidValue;
    gm_hcol<<<1, 64, 0, s>>>(hd, hs, H, m, j);
    return hipGetLastError();
}

hipError_t launch_gm_scale(const double* x, const double* h, double* y, int64_t n, hipStream_t s)
{
    gm_scale<<<blocks_for(n, 256), 256, 0, s>>>(x, h, y, n);
    return hipGetLastError();
}

hipError_t launch_gm_lsq(double* H, const double* beta, int m, double* y, hipStream_t s)
{
    if (m < 1 || m > GMRES_MAX_RESTART) return hipErrorInvalidValue;
    gm_lsq<<<1, 64, 0, s>>>(H, beta, m, y);
    return hipGetLastError();
}

hipError_t launch_residual(int jprec, const int64_t* rowptr, const int32_t* colidx, const int32_t* adj, int nc,
                           const void* A, const double* x, const double* b, double* r, int64_t n, int64_t nnz,
                           const uint8_t* mask, hipStream_t s)
{
    if (nodeblock_ok(adj, nc, A, x)) {
        launch_mv<1>(jprec, rowptr, adj, nc, A, x, b, r, n, nnz, s, nullptr, 0.0, mask);
    } else {
        const int bl = blocks_for(n * 16, 256);
        if (jprec == 64) residual_csr<double><<<bl, 256, 0, s>>>(rowptr, colidx, (const double*)A, x, b, r, n, mask);
        else residual_csr<float><<<bl, 256, 0, s>>>(rowptr, colidx, (const float*)A, x, b, r, n, mask);
    }
    return hipGetLastError();
}

hipError_t launch_smooth(int jprec, const int64_t* rowptr, const int32_t* colidx, const int32_t* adj, int nc,
                         const void* A, const double* x, const double* b, const double* Binv, double omega, double* r,
                         double* y, int64_t n, int64_t nnz, hipStream_t s)
{
    if (nodeblock_ok(adj, nc, A, x)) {
        launch_mv<2>(jprec, rowptr, adj, nc, A, x, b, y, n, nnz, s, Binv, omega);
        return hipGetLastError();
    }
    hipError_t e = launch_residual(jprec, rowptr, colidx, adj, nc, A, x, b, r, n, nnz, nullptr, s);
    if (e == hipSuccess) e = hipMemcpyAsync(y, x, sizeof(double) * n, hipMemcpyDeviceToDevice, s);
    if (e == hipSuccess) e = launch_bj_update(nc, Binv, r, y, omega, 0, n / nc, s);
    return e;
}

hipError_t launch_bj_update(int nc, const double* Binv, const double* r, double* x, double omega, int first,
                            int64_t nv, hipStream_t s)
{
    const int bl = blocks_for(nv, 256);
    if (nc == 3) bj_update<3><<<bl, 256, 0, s>>>(Binv, r, x, omega, first, nv);
    else bj_update<4><<<bl, 256, 0, s>>>(Binv, r, x, omega, first, nv);
    return hipGetLastError();
}

hipError_t launch_node_transfer(const int64_t* rowptr, const int32_t* colidx, const double* w, const double* x,
                                const double* base, const uint8_t* mask, double* y, int64_t nrows, int nc, hipStream_t s)
{
    node_transfer<<<blocks_for(nrows * nc, 256), 256, 0, s>>>(rowptr, colidx, w, x, base, mask, y, nrows, nc);
    return hipGetLastError();
}

hipError_t launch_inject(const int64_t* inj, const double* uf, double* uc, int64_t nvc, int nc, hipStream_t s)
{
    inject_state<<<blocks_for(nvc * nc, 256), 256, 0, s>>>(inj, uf, uc, nvc, nc);
    return hipGetLastError();
}

// two tableaux, two panels (G, flags, pivots), the pivoted flags, the pivot
// rows of all steps and, as its last word, the error flag
size_t dense_inverse_work_bytes(int n)
{
    const size_t m = (size_t)n;
    return sizeof(double) * (2 * m * m + 2 * m * GJ_BLOCK) + sizeof(int) * (2 * (m + GJ_BLOCK) + 2 * m + 2);
}

hipError_t launch_dense_inverse(int jprec, const int64_t* rowptr, const int32_t* colidx, const void* J, int n,
                                void* work, double* inv, int* err, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (n > MG_DENSE_MAX) return hipErrorInvalidValue;
    static_assert(MG_DENSE_MAX <= 3 * GJ_TPB, "gj_step is built for at most three rows per thread");
    const size_t nn = (size_t)n * n;
    double* M[2] = {(double*)work, (double*)work + nn};
    GJPanel G[2];
    G[0].G = M[1] + nn;
    G[1].G = G[0].G + (size_t)n * GJ_BLOCK;
    int* iw = (int*)(G[1].G + (size_t)n * GJ_BLOCK);
    for (int q = 0; q < 2; ++q) {
        G[q].flag = iw;
        G[q].piv = iw + n;
        iw += n + GJ_BLOCK;
    }
    int* done = iw;
    int* piv = done + n;
    if (jprec == 64) gj_load<double><<<n, 256, 0, s>>>(rowptr, colidx, (const double*)J, n, M[0], done, err);
    else gj_load<float><<<n, 256, 0, s>>>(rowptr, colidx, (const float*)J, n, M[0], done, err);
    // launch l applies panel l - 1 (none for l = 0) and factors panel l
    const int np = (n + GJ_BLOCK - 1) / GJ_BLOCK;
    const unsigned wgs = ((unsigned)np * np + GJ_TPB / 64 - 1) / (GJ_TPB / 64);
    for (int l = 0; l <= np; ++l) {
        const double* in = M[l > 0 ? (l - 1) & 1 : 0];
        double* out = M[l > 0 ? l & 1 : 1];
        const unsigned g = l > 0 ? 1 + wgs : 1;
        const int k0 = l > 0 ? (l - 1) * GJ_BLOCK : 0;
        const auto step = [&](auto kern) {
            kern<<<g, GJ_TPB, 0, s>>>(in, out, G[(l + 1) & 1], G[l & 1], done, piv, err, n, k0, l == 0);
        };
        switch ((n + GJ_TPB - 1) / GJ_TPB) {
        case 1: step(gj_step<1>); break;
        case 2: step(gj_step<2>); break;
        default: step(gj_step<3>); break;
        }
    }
    gj_unpermute<<<blocks_for((int64_t)n * n, 256), 256, 0, s>>>(M[np & 1], piv, n, inv);
    return hipGetLastError();
}

hipError_t launch_dense_matvec(const double* A, const double* x, double* y, int n, hipStream_t s)
{
    dense_matvec<<<blocks_for((int64_t)n * 64, 256), 256, 0, s>>>(A, x, y, n);
    return hipGetLastError();
}

}  // namespace nsfv1
