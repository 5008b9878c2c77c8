// Coarse level of the PCG preconditioner for one mesh: an additive
// two-level preconditioner M = M1 + P A_c^-1 P^T, with M1 the cluster block
// Jacobi and P the rigid-body modes (3 translations, 3 rotations about the
// centroid, orthonormal per aggregate) of aggregates of free vertices that
// are cells of a voxel grid over the current positions.  The PCG solves of
// the Newton iterations are ill-conditioned in the smooth, near-rigid motions
// of large pieces of the mesh (one iteration of block Jacobi moves
// information one block row); the coarse space removes those directly.
//
// Every few Newton iterations (coarse_setup): the free vertices are counted
// per voxel, voxels of many vertices (folded meshes, uneven ones) are split
// into pieces in vertex order, P is formed per aggregate (6 columns, a
// rotation direction dropped when its inertia is tiny), A_c = P^T A P is
// assembled with a fixed summation order (a stable radix sort of the blocks
// by aggregate pair, one workgroup per pair), and replaced by its inverse
// (blocked symmetric sweeps), all on the device; the host reads the box and
// the voxel counts and plans the aggregates.  In between, the level of
// the last build is reused: with an earlier system's A_c^-1 and P the
// preconditioner is still symmetric positive definite, only less exact.  Per PCG iteration (two
// kernels after the update): r_c = P^T r (one workgroup per aggregate), then
// per aggregate its rows of e_c = A_c^-1 r_c, their part of r_c . e_c and
// z += P e_c on its vertices (one workgroup per aggregate).  Since r . P e_c = r_c . e_c, the preconditioned dot of the
// iteration is the update's r . z1 plus those partials.
// Dirichlet vertices belong to no aggregate, so the coarse correction never
// moves them.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"
#include "linalg.hpp"
#include "prim.hpp"

namespace idp {

constexpr int COARSE_MAX_AGG = 320;  // aggregates at most (A_c of order 1920, 29 MB)

namespace {

// key of each block by the aggregate pair of its row and column; K * K (a
// run of its own, sorted last, then skipped) when either vertex is in no
// aggregate
__global__ void k_coarse_keys(long ne, const int* __restrict__ erow, const int* __restrict__ ecol, long nc,
                              const int* __restrict__ crow, const int* __restrict__ ccol, const int* __restrict__ agg,
                              int K, unsigned long long* __restrict__ key, unsigned* __restrict__ val)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ne + nc) return;
    const int r = i < ne ? erow[i] : crow[i - ne];
    const int c = i < ne ? ecol[i] : ccol[i - ne];
    const int ar = agg[r], ac = agg[c];
    key[i] = (ar < 0 || ac < 0) ? (unsigned long long)K * K : (unsigned long long)ar * K + ac;
    val[i] = (unsigned)i;
}

__global__ void k_coarse_heads(long n, const unsigned long long* __restrict__ key, unsigned* __restrict__ head)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    head[i] = (i < n && (i == 0 || key[i] != key[i - 1])) ? 1u : 0u;
}

// segment starts: seg[hs[i]] = i for each run head
__global__ void k_coarse_segs(long n, const unsigned* __restrict__ head, const unsigned* __restrict__ hs,
                              unsigned* __restrict__ seg)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !head[i]) return;
    seg[hs[i]] = (unsigned)i;
}

__global__ void k_coarse_fill(long n, double* __restrict__ a, double v)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// one workgroup per aggregate pair (grid-stride over the nseg pairs, counted
// on the device): sum of P_r^T A_rc P_c over its blocks (threads take every
// 256th block, then a fixed butterfly per wavefront and the wavefronts in
// order), into the dense column-major A_c of leading dimension ld.  A pair
// holds up to a few thousand blocks behind dependent loads: one wavefront per
// pair took 450 us on the 64x16x16 bar.
__global__ void __launch_bounds__(256) k_coarse_ac(const unsigned* __restrict__ nsegp, const unsigned* __restrict__ seg,
                                                   unsigned nrun, const unsigned long long* __restrict__ key,
                                                   const unsigned* __restrict__ val, long ne,
                                                   const int* __restrict__ erow, const int* __restrict__ ecol,
                                                   const double* __restrict__ evals, const int* __restrict__ crow,
                                                   const int* __restrict__ ccol, const double* __restrict__ cvals,
                                                   long nc, const double* __restrict__ P, int K, int lda,
                                                   double* __restrict__ Ac)
{
    __shared__ double sh[4][36];
    const unsigned nseg = *nsegp;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (unsigned sgi = blockIdx.x; sgi < nseg; sgi += gridDim.x) {
        const unsigned b0 = seg[sgi], b1 = sgi + 1 < nseg ? seg[sgi + 1] : nrun;
        const unsigned long long kk = key[b0];
        if (kk == (unsigned long long)K * K) continue;  // blocks outside the aggregates (uniform)
        double acc[36];
#pragma unroll
        for (int e = 0; e < 36; ++e) acc[e] = 0.0;
        for (unsigned j = b0 + threadIdx.x; j < b1; j += 256) {
            const long i = val[j];
            const bool el = i < ne;
            const long k = el ? i : i - ne;
            const int r = el ? erow[k] : crow[k];
            const int c = el ? ecol[k] : ccol[k];
            const double* vals = el ? evals : cvals;
            const long ld = el ? ne : nc;
            double a[9];
#pragma unroll
            for (int e = 0; e < 9; ++e) a[e] = vals[e * ld + k];
            const double* Pr = P + 18 * (size_t)r;
            const double* Pc = P + 18 * (size_t)c;
            double ap[18];  // A P_c, 3 x 6
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int m = 0; m < 6; ++m)
                    ap[6 * q + m] = a[3 * q] * Pc[m] + a[3 * q + 1] * Pc[6 + m] + a[3 * q + 2] * Pc[12 + m];
#pragma unroll
            for (int l = 0; l < 6; ++l)
#pragma unroll
                for (int m = 0; m < 6; ++m)
                    acc[6 * l + m] += Pr[l] * ap[m] + Pr[6 + l] * ap[6 + m] + Pr[12 + l] * ap[12 + m];
        }
#pragma unroll
        for (int e = 0; e < 36; ++e) {
            double v = acc[e];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            if (lane == 0) sh[wave][e] = v;
        }
        __syncthreads();
        if (threadIdx.x < 36) {
            const int ar = (int)(kk / (unsigned long long)K), ac = (int)(kk % (unsigned long long)K);
            const int l = threadIdx.x / 6, m = threadIdx.x % 6;
            double v = 0.0;
#pragma unroll
            for (int w = 0; w < 4; ++w) v += sh[w][threadIdx.x];
            Ac[(size_t)(6 * ar + l) + (size_t)(6 * ac + m) * lda] = v;
        }
        __syncthreads();
    }
}

// dofs of dropped modes (zero rows) and of the padding: 1 on the diagonal
__global__ void k_coarse_diag(int n, double* __restrict__ Ac)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && Ac[(size_t)i * n + i] == 0.0) Ac[(size_t)i * n + i] = 1.0;
}

// ---- inverse of A_c by blocked symmetric sweeps --------------------------
// Sweeping block k of a symmetric matrix: B_kk = -A_kk^-1, B_ik = A_ik A_kk^-1,
// B_ij = A_ij - A_ik A_kk^-1 A_kj; after all blocks B = -A^-1, symmetric
// throughout, so only the lower tiles are formed.  A_kk^-1 = T^T T enters by
// T = L^-1 of the tile's Cholesky factor, B_ij = A_ij - U_i^T U_j with
// U_j = T A_kj: what is left of the matrix is then the Cholesky one, with its
// error (a stiff contact gives A_c a condition of 1e12; with A_kk^-1 itself
// the error was 1,000 times a Cholesky inverse's there, pivots went negative
// and the level was refused).  One launch per block of SW rows, one workgroup
// per lower tile, reading one copy of the matrix and writing the other; the
// workgroup of the next diagonal tile also factors it, so a launch is the whole
// serial step.  (A library Cholesky and inverse took 2.2 ms of small dependent
// kernels at order 780 and 5 ms at 1,900.)
constexpr int SW = 64;
constexpr int SW_LD = SW + 1;

// M (SW x SW, symmetric positive definite, in LDS) -> T = L^-1, M = L L^T.
// Row operations that eliminate below each pivot, with the unit lower factor's
// inverse growing in place of the eliminated columns, then each row by the root
// of its pivot.  Each thread keeps a 4 x 4 piece; four pivot rows at a time go
// through rows, and every thread brings its columns of them up to date by
// itself (with a barrier per pivot the 24 sweeps of order 1,536 took 8 us more
// each; 51 us now, as with A_kk^-1 in T's place).
// *ok: every pivot was positive.
__device__ inline void sweep_factor(double (*M)[SW_LD], double (*rows)[4][SW], int* ok)
{
#pragma clang fp contract(fast)
    const int ti = (threadIdx.x >> 4) * 4, tj = (threadIdx.x & 15) * 4;
    double a[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) a[i][j] = M[ti + i][tj + j];
    bool good = true;
    for (int p = 0; p < SW; p += 4) {
        double(*r)[SW] = rows[(p >> 2) & 1];
        if (ti == p) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) r[i][tj + j] = a[i][j];
        }
        __syncthreads();
        double P[4][4], R[4][4], F[4][4];  // the pivot rows in the pivot, this thread's and (below: by symmetry) its rows' columns
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                P[q][j] = r[q][p + j];
                R[q][j] = r[q][tj + j];
                F[q][j] = r[q][ti + j];
            }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double d = P[q][q];
            good = good && d > 0;
            const double id = 1.0 / d;
            // the block's later pivot rows
#pragma unroll
            for (int b = q + 1; b < 4; ++b) {
                const double f = P[q][b] * id;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (j > q) P[b][j] = P[b][j] - f * P[q][j];
                    R[b][j] = tj + j == p + q ? -f : R[b][j] - f * R[q][j];
                    F[b][j] = F[b][j] - f * F[q][j];
                }
            }
            // this thread's rows below the block
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double f = F[q][i] * id;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const double t = tj + j == p + q ? -f : a[i][j] - f * R[q][j];
                    a[i][j] = ti > p ? t : a[i][j];
                }
            }
        }
        if (ti == p)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) a[i][j] = R[i][j];
    }
    __syncthreads();
    double* piv = rows[0][0];
    if (ti == tj)
#pragma unroll
        for (int i = 0; i < 4; ++i) piv[ti + i] = a[i][i];  // the pivots
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const double s = 1.0 / sqrt(piv[ti + i]);
#pragma unroll
        for (int j = 0; j < 4; ++j) M[ti + i][tj + j] = tj + j < ti + i ? a[i][j] * s : tj + j == ti + i ? s : 0.0;
    }
    if (!good && threadIdx.x == 0) *ok = 0;
    __syncthreads();
}

// tile (i, j) of the symmetric matrix stored by its lower tiles, into LDS
__device__ inline void sweep_load(const double* __restrict__ A, int n, int i, int j, double (*T)[SW_LD])
{
    const int x = threadIdx.x & 63, y0 = threadIdx.x >> 6;
    if (i >= j) {  // column-major: x along the rows of a column
        for (int y = y0; y < SW; y += 4) T[x][y] = A[(size_t)(SW * j + y) * n + SW * i + x];
    } else {
        for (int y = y0; y < SW; y += 4) T[y][x] = A[(size_t)(SW * i + y) * n + SW * j + x];
    }
}

__device__ inline void sweep_put(const double (*c)[4], double (*T)[SW_LD])
{
    const int ti = (threadIdx.x >> 4) * 4, tj = (threadIdx.x & 15) * 4;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) T[ti + u][tj + v] = c[u][v];
}

// C (4 x 4 per thread) = X Y, or X^T Y (TX), both SW x SW in LDS, over the
// inner indices [k0, k1): the rest is zero where X is the lower triangle T
template <bool TX>
__device__ inline void sweep_mul(const double (*X)[SW_LD], const double (*Y)[SW_LD], int k0, int k1, double (*c)[4])
{
#pragma clang fp contract(fast)
    const int ti = (threadIdx.x >> 4) * 4, tj = (threadIdx.x & 15) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) c[i][j] = 0.0;
#pragma unroll 4
    for (int k = k0; k < k1; ++k) {
        double x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u] = TX ? X[k][ti + u] : X[ti + u][k];
            y[u] = Y[k][tj + u];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) c[i][j] += x[i] * y[j];
    }
}

// T of the first diagonal tile
__global__ void __launch_bounds__(256) k_coarse_first(int n, const double* __restrict__ A, double* __restrict__ D,
                                                      int* __restrict__ info)
{
    __shared__ double M[SW][SW_LD], rows[2][4][SW];
    __shared__ int ok;
    if (threadIdx.x == 0) ok = 1;
    sweep_load(A, n, 0, 0, M);
    __syncthreads();
    sweep_factor(M, rows, &ok);
    for (int e = threadIdx.x; e < SW * SW; e += 256) D[e] = M[e / SW][e % SW];
    if (threadIdx.x == 0) *info = ok ? 0 : 1;
}

// sweep of block k: src -> dst; D = T of the block, Dn receives the next one.
// The last sweep (k = n / SW - 1) writes the inverse itself, both triangles.
__global__ void __launch_bounds__(256) k_coarse_sweep(int n, int k, const double* __restrict__ src,
                                                      double* __restrict__ dst, const double* __restrict__ D,
                                                      double* __restrict__ Dn, int* __restrict__ info)
{
    __shared__ double X[SW][SW_LD], Y[SW][SW_LD], rows[2][4][SW];
    __shared__ int ok;
    const int nt = n / SW;
    int i = (int)((sqrt(8.0 * blockIdx.x + 1.0) - 1.0) / 2.0);
    while ((i + 1) * (i + 2) / 2 <= (int)blockIdx.x) ++i;
    while (i * (i + 1) / 2 > (int)blockIdx.x) --i;
    const int j = (int)blockIdx.x - i * (i + 1) / 2;  // lower tile (i, j)
    const int ti = (threadIdx.x >> 4) * 4, tj = (threadIdx.x & 15) * 4;
    const int r0 = 16 * (threadIdx.x >> 6), r1 = r0 + 16;  // the wavefront's rows: T is zero right of, T^T left of them
    const bool last = k == nt - 1;
    const double sg = last ? -1.0 : 1.0;
    if (threadIdx.x == 0) ok = 1;
    for (int e = threadIdx.x; e < SW * SW; e += 256) X[e / SW][e % SW] = D[e];
    double c[4][4];
    const bool trans = j == k && i != k;  // c holds the transpose of the tile
    if (i == k && j == k) {
        __syncthreads();
        sweep_mul<true>(X, X, r0, SW, c);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) c[u][v] = -c[u][v];
    } else {
        sweep_load(src, n, k, trans ? i : j, Y);
        __syncthreads();
        sweep_mul<false>(X, Y, 0, r1, c);  // U of the tile's column (row, for j == k)
        if (i == k || j == k) {
            __syncthreads();
            sweep_put(c, Y);
            __syncthreads();
            sweep_mul<true>(X, Y, r0, SW, c);  // A_kk^-1 A_kj
        } else {
            double u[4][4];
            if (i != j) {
                __syncthreads();
                sweep_load(src, n, k, i, Y);
                __syncthreads();
                sweep_mul<false>(X, Y, 0, r1, u);
            }
            __syncthreads();
            sweep_put(c, Y);
            if (i != j) sweep_put(u, X);
            else sweep_put(c, X);
            __syncthreads();
            sweep_mul<true>(X, Y, 0, SW, c);
            __syncthreads();
            sweep_load(src, n, i, j, X);
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) c[u][v] = X[ti + u][tj + v] - c[u][v];
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (trans) X[tj + v][ti + u] = c[u][v];
            else X[ti + u][tj + v] = c[u][v];
        }
    __syncthreads();
    const int x = threadIdx.x & 63, y0 = threadIdx.x >> 6;
    for (int y = y0; y < SW; y += 4) {
        // the diagonal tile from its lower triangle, so that the result is exactly symmetric
        const double v = i == j && x < y ? X[y][x] : X[x][y];
        dst[(size_t)(SW * j + y) * n + SW * i + x] = sg * v;
    }
    if (last && i != j)
        for (int y = y0; y < SW; y += 4) dst[(size_t)(SW * i + y) * n + SW * j + x] = sg * X[y][x];
    if (i == k + 1 && j == k + 1) {
        __syncthreads();
        sweep_factor(X, rows, &ok);
        for (int e = threadIdx.x; e < SW * SW; e += 256) Dn[e] = X[e / SW][e % SW];
        if (threadIdx.x == 0 && !ok) *info = 1;
    }
}

// ---- aggregates -----------------------------------------------------------
// box and number of the free vertices, per block (7 doubles each)
__global__ void __launch_bounds__(256) k_coarse_box(int nV, const double* __restrict__ X,
                                                    const unsigned char* __restrict__ fixed, double* __restrict__ part)
{
    __shared__ double sh[4][7];
    double b[7] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300, 0.0};
    for (int v = blockIdx.x * 256 + threadIdx.x; v < nV; v += 256 * gridDim.x) {
        if (fixed && fixed[v]) continue;
        b[6] += 1.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            b[d] = fmin(b[d], X[3 * (size_t)v + d]);
            b[3 + d] = fmax(b[3 + d], X[3 * (size_t)v + d]);
        }
    }
#pragma unroll
    for (int e = 0; e < 7; ++e) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double t = __shfl_xor(b[e], o, 64);
            b[e] = e < 3 ? fmin(b[e], t) : e < 6 ? fmax(b[e], t) : b[e] + t;
        }
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][e] = b[e];
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        const int e = threadIdx.x;
        double r = sh[0][e];
        for (int w = 1; w < 4; ++w) r = e < 3 ? fmin(r, sh[w][e]) : e < 6 ? fmax(r, sh[w][e]) : r + sh[w][e];
        part[7 * blockIdx.x + e] = r;
    }
}

struct CoarseGrid {
    double lo[3], h;
    int n[3];
};

// voxel of every free vertex (ncell for the others) and the vertices per voxel
__global__ void k_coarse_cells(int nV, const double* __restrict__ X, const unsigned char* __restrict__ fixed,
                               CoarseGrid g, unsigned ncell, unsigned* __restrict__ key, unsigned* __restrict__ vert,
                               unsigned* __restrict__ cnt)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV) return;
    unsigned k = ncell;
    if (!(fixed && fixed[v])) {
        int c[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) c[d] = min(max((int)floor((X[3 * (size_t)v + d] - g.lo[d]) / g.h), 0), g.n[d] - 1);
        k = (unsigned)c[0] + (unsigned)g.n[0] * ((unsigned)c[1] + (unsigned)g.n[1] * (unsigned)c[2]);
        atomicAdd(cnt + k, 1u);
    }
    key[v] = k;
    vert[v] = (unsigned)v;
}

__global__ void k_coarse_zero(long n, unsigned* __restrict__ a)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0u;
}

// symmetric 3x3 eigen-decomposition by cyclic Jacobi (columns of V)
__device__ inline void eig3(double* a, double* w, double* V)
{
    for (int i = 0; i < 9; ++i) V[i] = (i % 4 == 0) ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 50; ++sweep) {
        const double off = a[1] * a[1] + a[2] * a[2] + a[5] * a[5];
        if (off < 1e-300) break;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = p + 1; q < 3; ++q) {
                const double apq = a[3 * p + q];
                if (apq == 0.0) continue;
                const double th = (a[3 * q + q] - a[3 * p + p]) / (2 * apq);
                const double t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1));
                const double c = 1 / sqrt(t * t + 1), s = t * c;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const double x = a[3 * k + p], y = a[3 * k + q];
                    a[3 * k + p] = c * x - s * y;
                    a[3 * k + q] = s * x + c * y;
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const double x = a[3 * p + k], y = a[3 * q + k];
                    a[3 * p + k] = c * x - s * y;
                    a[3 * q + k] = s * x + c * y;
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const double x = V[3 * k + p], y = V[3 * k + q];
                    V[3 * k + p] = c * x - s * y;
                    V[3 * k + q] = s * x + c * y;
                }
            }
    }
    for (int i = 0; i < 3; ++i) w[i] = a[4 * i];
}

// one workgroup per aggregate: centroid, inertia, and the 6 columns of P for
// its vertices (3 translations, 3 rotations scaled by w_k^(-1/2), tiny
// inertia dropped), by vertex (P, for A_c) and by slot in planes (Ps)
__global__ void __launch_bounds__(256) k_coarse_modes(const int* __restrict__ aptr, const unsigned* __restrict__ avert,
                                                      const double* __restrict__ X, int nfree, int* __restrict__ agg,
                                                      int* __restrict__ av, double* __restrict__ P,
                                                      double* __restrict__ Ps)
{
    __shared__ double sh[4][6], cen[3], Rs[9];
    const int a = blockIdx.x, j0 = aptr[a], j1 = aptr[a + 1], n = j1 - j0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto sum = [&](double* acc, int N) {  // totals over the workgroup, left in sh[0] by thread order
        for (int m = 0; m < N; ++m) {
            double v = acc[m];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            if (lane == 0) sh[wave][m] = v;
        }
        __syncthreads();
        for (int m = 0; m < N; ++m) acc[m] = ((sh[0][m] + sh[1][m]) + sh[2][m]) + sh[3][m];
        __syncthreads();
    };
    double c[6] = {0, 0, 0, 0, 0, 0};
    for (int j = j0 + (int)threadIdx.x; j < j1; j += 256)
        for (int d = 0; d < 3; ++d) c[d] += X[3 * (size_t)avert[j] + d];
    sum(c, 3);
    if (threadIdx.x < 3) cen[threadIdx.x] = (threadIdx.x == 0 ? c[0] : threadIdx.x == 1 ? c[1] : c[2]) / n;
    __syncthreads();
    double J[6] = {0, 0, 0, 0, 0, 0};  // xx, xy, xz, yy, yz, zz of |d|^2 I - d d^T
    for (int j = j0 + (int)threadIdx.x; j < j1; j += 256) {
        const size_t v = avert[j];
        const double d0 = X[3 * v] - cen[0], d1 = X[3 * v + 1] - cen[1], d2 = X[3 * v + 2] - cen[2];
        J[0] += d1 * d1 + d2 * d2;
        J[1] -= d0 * d1;
        J[2] -= d0 * d2;
        J[3] += d0 * d0 + d2 * d2;
        J[4] -= d1 * d2;
        J[5] += d0 * d0 + d1 * d1;
    }
    sum(J, 6);
    if (threadIdx.x == 0) {
        double A[9] = {J[0], J[1], J[2], J[1], J[3], J[4], J[2], J[4], J[5]}, w[3], V[9];
        eig3(A, w, V);
        const double wmax = fmax(w[0], fmax(w[1], w[2]));
        for (int k = 0; k < 3; ++k) {
            const double sc = (wmax > 0 && w[k] > 1e-10 * wmax) ? 1.0 / sqrt(w[k]) : 0.0;
            for (int p = 0; p < 3; ++p) Rs[3 * p + k] = V[3 * p + k] * sc;
        }
    }
    __syncthreads();
    const double tn = 1.0 / sqrt((double)n);
    for (int j = j0 + (int)threadIdx.x; j < j1; j += 256) {
        const int v = (int)avert[j];
        const double d[3] = {X[3 * (size_t)v] - cen[0], X[3 * (size_t)v + 1] - cen[1], X[3 * (size_t)v + 2] - cen[2]};
        double Pv[18];
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int m = 0; m < 3; ++m) Pv[6 * q + m] = q == m ? tn : 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {  // rotation about axis u: u x d
            const double u[3] = {Rs[k], Rs[3 + k], Rs[6 + k]};
            Pv[3 + k] = u[1] * d[2] - u[2] * d[1];
            Pv[6 + 3 + k] = u[2] * d[0] - u[0] * d[2];
            Pv[12 + 3 + k] = u[0] * d[1] - u[1] * d[0];
        }
        agg[v] = a;
        av[j] = v;
#pragma unroll
        for (int q = 0; q < 18; ++q) {
            P[18 * (size_t)v + q] = Pv[q];
            Ps[(size_t)q * nfree + j] = Pv[q];
        }
    }
}

__global__ void k_coarse_none(int nV, int* __restrict__ agg)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < nV) agg[v] = -1;
}

}  // namespace

// ---------------------------------------------------------------------------
// per PCG iteration
// ---------------------------------------------------------------------------
constexpr int COARSE_BLOCK = 256;

// fixed-order sum of N values over a workgroup of COARSE_BLOCK threads:
// xor butterfly per wavefront, then the wavefronts in order (all threads
// get the totals)
template <int N>
__device__ inline void coarse_block_sum(double* acc, double (*sh)[N])
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int m = 0; m < N; ++m) {
        double v = acc[m];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        acc[m] = v;
    }
    if (lane == 0)
#pragma unroll
        for (int m = 0; m < N; ++m) sh[w][m] = acc[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < COARSE_BLOCK / 64; ++k) v += sh[k][m];
        acc[m] = v;
    }
}

// r_c = P^T r: one workgroup per aggregate over its vertex list
__global__ void __launch_bounds__(COARSE_BLOCK) k_coarse_restrict(int K, int nfree, const int* __restrict__ aptr,
                                                                  const int* __restrict__ avert,
                                                                  const double* __restrict__ Ps,
                                                                  const double* __restrict__ r,
                                                                  const int* __restrict__ flag,
                                                                  double* __restrict__ rc)
{
    __shared__ double sh[COARSE_BLOCK / 64][6];
    const int a = blockIdx.x;
    if (*(volatile const int*)flag != 0) return;  // uniform over the grid
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int j = aptr[a] + (int)threadIdx.x; j < aptr[a + 1]; j += COARSE_BLOCK) {
        const int v = avert[j];
        double Pv[18];
#pragma unroll
        for (int m = 0; m < 18; ++m) Pv[m] = Ps[(size_t)m * nfree + j];
        const double r0 = r[3 * v], r1 = r[3 * v + 1], r2 = r[3 * v + 2];
#pragma unroll
        for (int m = 0; m < 6; ++m) acc[m] += Pv[m] * r0 + Pv[6 + m] * r1 + Pv[12 + m] * r2;
    }
    coarse_block_sum<6>(acc, sh);
    if (threadIdx.x < 6) {
        double v = acc[0];
#pragma unroll
        for (int m = 1; m < 6; ++m) v = (int)threadIdx.x == m ? acc[m] : v;
        rc[6 * a + threadIdx.x] = v;
    }
}

// one workgroup per aggregate a: e = rows 6a..6a+5 of A_c^-1 times r_c, the
// partial r_c . e_c of those rows, and z += P_v e for the vertices of a
__global__ void __launch_bounds__(COARSE_BLOCK) k_coarse_solve(int K, int ncd, int lda, int nfree, const int* __restrict__ aptr,
                                                               const int* __restrict__ avert,
                                                               const double* __restrict__ Ps,
                                                               const double* __restrict__ Ainv,
                                                               const double* __restrict__ rc,
                                                               const int* __restrict__ flag,
                                                               double* __restrict__ part, double* __restrict__ z)
{
    __shared__ double sh[COARSE_BLOCK / 64][6];
    const int a = blockIdx.x;
    if (*(volatile const int*)flag != 0) return;  // uniform over the grid
    double e[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const double* A0 = Ainv + (size_t)(6 * a) * lda;  // symmetric: rows = columns
    // eight columns' loads in flight at once; each thread still adds its
    // columns in increasing order
    constexpr int U = 8;
    int j = threadIdx.x;
    for (; j + (U - 1) * COARSE_BLOCK < ncd; j += U * COARSE_BLOCK) {
        double rj[U], av[U][6];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            rj[u] = rc[j + u * COARSE_BLOCK];
#pragma unroll
            for (int m = 0; m < 6; ++m) av[u][m] = A0[(size_t)m * lda + j + u * COARSE_BLOCK];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < 6; ++m) e[m] += av[u][m] * rj[u];
    }
    for (; j < ncd; j += COARSE_BLOCK) {
        const double rj = rc[j];
#pragma unroll
        for (int m = 0; m < 6; ++m) e[m] += A0[(size_t)m * lda + j] * rj;
    }
    coarse_block_sum<6>(e, sh);
    if (threadIdx.x == 0) {
        double d = 0.0;
#pragma unroll
        for (int m = 0; m < 6; ++m) d += rc[6 * a + m] * e[m];
        part[a] = d;
    }
    for (int j = aptr[a] + (int)threadIdx.x; j < aptr[a + 1]; j += COARSE_BLOCK) {
        const int v = avert[j];
        double Pv[18];
#pragma unroll
        for (int m = 0; m < 18; ++m) Pv[m] = Ps[(size_t)m * nfree + j];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            double s = 0.0;
#pragma unroll
            for (int m = 0; m < 6; ++m) s += Pv[6 * q + m] * e[m];
            z[3 * v + q] += s;
        }
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
bool coarse_setup(LinWork& L, hipStream_t s, const MeshDev& m, const double* X)
{
    CoarseWork& C = L.coarse;
    const int nV = m.nV;
    if (C.verts_per_agg <= 0 || m.inst.B != 1 || !X || nV < 2 * C.verts_per_agg) return false;
    if (C.ready && C.age < C.rebuild_every && C.nV == nV && C.mask == m.proj_mask()) {
        ++C.age;  // the level of an earlier system of this mesh
        return true;
    }
    C.ready = false;
    // box of the free vertices
    const int nbox = std::min(grid_for(nV, 256), 64);
    double* dbox = C.box.ensure(7 * (size_t)nbox, s);
    IDP_LAUNCH(k_coarse_box, nbox, 256, 0, s, nV, X, m.proj_mask(), dbox);
    double* hb = L.pin->as<double>(7 * (size_t)nbox);
    IDP_HIP(hipMemcpyAsync(hb, dbox, 7 * (size_t)nbox * sizeof(double), hipMemcpyDeviceToHost, s));
    IDP_HIP(hipStreamSynchronize(s));
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    long nfree = 0;
    for (int b = 0; b < nbox; ++b) {
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], hb[7 * b + d]);
            hi[d] = std::max(hi[d], hb[7 * b + 3 + d]);
        }
        nfree += (long)hb[7 * b + 6];
    }
    if (nfree < 2 * C.verts_per_agg) return false;
    for (int d = 0; d < 3; ++d)
        if (!(hi[d] - lo[d] < 1e150)) return false;  // not a mesh that can be binned
    // voxel edge for about nfree / verts_per_agg voxels over the box; a
    // direction thinner than a quarter of the edge (a sheet) counts as one
    // voxel: its volume would ask for far more voxels than that
    const double target = std::min((double)nfree / C.verts_per_agg, (double)COARSE_MAX_AGG);
    double ext[3] = {hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]};
    std::sort(ext, ext + 3);
    double hcell = 0.0;
    for (int nd = 3; nd > 0; --nd) {
        double vol = 1.0;
        for (int d = 3 - nd; d < 3; ++d) vol *= ext[d];
        hcell = std::pow(vol / target, 1.0 / nd);
        if (hcell > 0 && hcell <= 4 * ext[3 - nd]) break;
    }
    if (!(hcell > 0)) return false;
    // vertices per voxel; larger voxels while there are too many of them
    constexpr unsigned MAX_CELLS = 65536;
    unsigned* key = C.cells.ensure(4 * (size_t)nV + MAX_CELLS, s);
    unsigned* vert = key + nV;
    std::vector<unsigned> cnt;
    CoarseGrid g;
    unsigned ncell = 0;
    int K = 0;
    for (int pass = 0; pass < 8; ++pass) {
        double cells = 1.0;
        for (int d = 0; d < 3; ++d) {
            g.lo[d] = lo[d];
            const double nd = std::floor((hi[d] - lo[d]) / hcell) + 1.0;
            cells *= nd;
            g.n[d] = (int)std::min(nd, 1e9);
        }
        g.h = hcell;
        if (cells > MAX_CELLS) {
            hcell *= std::cbrt(cells / MAX_CELLS) * 1.05;
            continue;
        }
        ncell = (unsigned)cells;
        unsigned* dc = key + 4 * (size_t)nV;
        IDP_LAUNCH(k_coarse_zero, grid_for(ncell, 256), 256, 0, s, (long)ncell, dc);
        IDP_LAUNCH(k_coarse_cells, grid_for(nV, 256), 256, 0, s, nV, X, m.proj_mask(), g, ncell, key, vert, dc);
        unsigned* hc = L.pin->as<unsigned>(ncell);
        IDP_HIP(hipMemcpyAsync(hc, dc, ncell * sizeof(unsigned), hipMemcpyDeviceToHost, s));
        IDP_HIP(hipStreamSynchronize(s));
        cnt.assign(hc, hc + ncell);
        K = 0;
        for (unsigned q : cnt) K += q > 0;
        if (K <= COARSE_MAX_AGG) break;
        hcell *= std::cbrt((double)K / COARSE_MAX_AGG) * 1.05;
    }
    if (K > COARSE_MAX_AGG || K < 1) return false;
    // a voxel of more than `cap` vertices, four times the size asked for, is cut
    // into pieces of equal size in vertex order, while the total stays bounded
    // (cutting at 256 saves 1-6% of a bar's iterations and 1-2% of its solve, but
    // gives ordinary voxels of small bars other aggregates than whole ones)
    auto pieces = [](unsigned n, double cap) { return (int)std::ceil(n / cap); };
    double cap = 4.0 * C.verts_per_agg;
    for (;; cap *= 1.25) {
        long k = 0;
        for (unsigned q : cnt) k += pieces(q, cap);
        if (k <= COARSE_MAX_AGG) {
            K = (int)k;
            break;
        }
    }
    if (K < 2) return false;
    std::vector<int> aptr;
    aptr.reserve(K + 1);
    long at = 0;
    for (unsigned q : cnt) {
        const int np = pieces(q, cap);
        for (int u = 0; u < np; ++u) aptr.push_back((int)(at + (long)q * u / np));
        at += q;
    }
    aptr.push_back((int)at);
    const int ncd = 6 * K, n = (ncd + SW - 1) / SW * SW;
    C.K = K;
    C.ncd = ncd;
    C.lda = n;
    C.nfree = (int)nfree;
    C.aptr.upload(aptr.data(), aptr.size(), s);
    // vertices by voxel, in vertex order (Dirichlet ones last), and the modes
    unsigned* key1 = key + 2 * (size_t)nV;
    unsigned* vert1 = key + 3 * (size_t)nV;
    int cbits = 1;
    while (cbits < 31 && (ncell >> cbits)) ++cbits;
    sort_pairs(s, C.tmp, key, key1, vert, vert1, nV, cbits);
    int* d_agg = C.agg.ensure(nV, s);
    int* d_av = C.avert.ensure(nfree, s);
    double* d_P = C.P.ensure(18 * (size_t)nV, s);
    double* d_Ps = C.Ps.ensure(18 * (size_t)nfree, s);
    IDP_LAUNCH(k_coarse_none, grid_for(nV, 256), 256, 0, s, nV, d_agg);
    IDP_LAUNCH(k_coarse_modes, K, 256, 0, s, C.aptr.p, vert1, X, (int)nfree, d_agg, d_av, d_P, d_Ps);
    // A_c = P^T A P, summed per aggregate pair in block order
    const long ne = m.nnzb_e, nc = L.ncb, nb = ne + nc;
    unsigned long long* k0 = C.key0.ensure(nb + 1, s);
    unsigned* v0 = C.val0.ensure(nb + 1, s);
    IDP_LAUNCH(k_coarse_keys, grid_for(nb, 256), 256, 0, s, ne, L.erow.p, m.e_col.p, nc, L.crow.p, L.ccol.p, d_agg, K,
               k0, v0);
    unsigned long long* k1 = C.key1.ensure(nb + 1, s);
    unsigned* v1 = C.val1.ensure(nb + 1, s);
    int kbits = 1;
    while (kbits < 63 && ((unsigned long long)K * K >> kbits)) ++kbits;
    sort_pairs(s, C.tmp, k0, k1, v0, v1, nb, kbits);
    unsigned* head = C.head.ensure(nb + 1, s);
    unsigned* hs = C.hs.ensure(nb + 1, s);
    IDP_LAUNCH(k_coarse_heads, grid_for(nb + 1, 256), 256, 0, s, nb, k1, head);
    excl_scan<unsigned>(s, C.tmp, head, hs, nb + 1);
    const long maxseg = std::min<long>(nb, (long)K * K + 1);
    unsigned* seg = C.seg.ensure(maxseg + 1, s);
    IDP_LAUNCH(k_coarse_segs, grid_for(nb, 256), 256, 0, s, nb, head, hs, seg);
    double* A0 = C.Ainv.ensure((size_t)n * n, s);
    double* A1 = C.Awork.ensure((size_t)n * n, s);
    const int nt = n / SW;
    double *src = A0, *dst = A1;
    if (nt & 1) std::swap(src, dst);  // nt sweeps end in Ainv
    IDP_LAUNCH(k_coarse_fill, grid_for((long)n * n, 256), 256, 0, s, (long)n * n, src, 0.0);
    IDP_LAUNCH(k_coarse_ac, (int)std::min<long>(maxseg, 4096), 256, 0, s, hs + nb, seg, (unsigned)nb, k1, v1, ne,
               L.erow.p, m.e_col.p, L.evals.p, L.crow.p, L.ccol.p, L.cvals.p, nc, d_P, K, n, src);
    IDP_LAUNCH(k_coarse_diag, grid_for(n, 256), 256, 0, s, n, src);
    // its inverse
    int* info = C.info.ensure(1, s);
    double* D = C.diag.ensure(2 * SW * SW, s);
    IDP_LAUNCH(k_coarse_first, 1, 256, 0, s, n, src, D, info);
    for (int k = 0; k < nt; ++k) {
        IDP_LAUNCH(k_coarse_sweep, nt * (nt + 1) / 2, 256, 0, s, n, k, src, dst, D + (k & 1) * SW * SW,
                   D + ((k + 1) & 1) * SW * SW, info);
        std::swap(src, dst);
    }
    int* hinfo = L.pin->as<int>(1);
    IDP_HIP(hipMemcpyAsync(hinfo, info, sizeof(int), hipMemcpyDeviceToHost, s));
    IDP_HIP(hipStreamSynchronize(s));
    if (*hinfo != 0) return false;  // not positive definite: no coarse level this time
    C.rc.ensure(ncd, s);
    C.nsb = K;  // one partial of r_c . e_c per aggregate
    C.part.ensure(2 * (size_t)C.nsb + 2, s);
    C.ready = true;
    C.age = 1;
    C.nV = nV;
    C.mask = m.proj_mask();
    return true;
}

void coarse_apply(LinWork& L, hipStream_t s, int nV, const double* r, double* z, const int* flag, int parity)
{
    (void)nV;
    CoarseWork& C = L.coarse;
    IDP_LAUNCH(k_coarse_restrict, C.K, COARSE_BLOCK, 0, s, C.K, C.nfree, C.aptr.p, C.avert.p, C.Ps.p, r, flag, C.rc.p);
    IDP_LAUNCH(k_coarse_solve, C.K, COARSE_BLOCK, 0, s, C.K, C.ncd, C.lda, C.nfree, C.aptr.p, C.avert.p, C.Ps.p, C.Ainv.p, C.rc.p,
               flag, C.part.p + (size_t)parity * C.nsb, z);
}

}  // namespace idp
