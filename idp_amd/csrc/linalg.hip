// Assembly of the projected Hessian into 3x3-block BSR and its solve.
//   triplets -> CSR, += M     Library/Math/CSR_MATRIX.h:49-56, INC_POTENTIAL.h:382-386
//   DBC projection            Library/Math/CSR_MATRIX.h:130-141
//   Newton direction solve    Library/Math/DIRECT_SOLVER.h:14-89 (replaced by PCG)
//
// The system is H = E + C: E has the static tet pattern (plus the lumped
// mass on the diagonal) and is refilled every Newton iteration by a gather
// over precomputed per-block contribution lists; C holds the contact blocks
// of the current constraint set, built by radix-sorting (row,col) keys of all
// local blocks and reducing each run in sort order.  Every sum has a fixed
// order, so results are bitwise reproducible.  PCG is preconditioned by block
// Jacobi over clusters of up to four vertices, for one mesh with a coarse level
// (coarse.hip); its dot products are deterministic two-level reductions whose
// final sum is recomputed by each consumer block.
#include "common.hpp"
#include "prim.hpp"
#include "kernels.hpp"
#include "linalg.hpp"

namespace idp {

// ---------------------------------------------------------------------------
// elastic BSR values and gradient gather
// ---------------------------------------------------------------------------
__global__ void k_elastic_values(long nnzb, const int* __restrict__ rowof, const int* __restrict__ col,
                                 const int* __restrict__ sptr, const int* __restrict__ src,
                                 const double* __restrict__ Hl, const double* __restrict__ mass,
                                 const int* __restrict__ vinst, const unsigned char* __restrict__ act,
                                 double* __restrict__ val)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnzb) return;
    if (act && !act[vinst[rowof[k]]]) return;  // instance not iterating
    double acc[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) acc[i] = 0.0;
    for (int j = sptr[k]; j < sptr[k + 1]; ++j) {
        const double* h = Hl + 9 * (size_t)src[j];
#pragma unroll
        for (int i = 0; i < 9; ++i) acc[i] += h[i];
    }
    int r = rowof[k];
    if (r == col[k]) {
        double m = mass[r];
        acc[0] += m;
        acc[4] += m;
        acc[8] += m;
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) val[i * (size_t)nnzb + k] = acc[i];  // component planes
}

// g_v = elastic (sum over incident tets) + M (x - x~) + barrier (sum over the
// contact diagonal run of v); DBC rows zeroed; rhs = -g
__global__ void k_gradient_gather(int nV, const int* __restrict__ ediag, const int* __restrict__ sptr,
                                  const int* __restrict__ src, const double* __restrict__ gl,
                                  const double* __restrict__ X, const double* __restrict__ Xt,
                                  const double* __restrict__ mass, const int* __restrict__ cdiag,
                                  const unsigned* __restrict__ cseg, const unsigned* __restrict__ cval,
                                  const double* __restrict__ gb, const unsigned char* __restrict__ dbc,
                                  const int* __restrict__ vinst, const unsigned char* __restrict__ act,
                                  double* __restrict__ g, double* __restrict__ rhs)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV) return;
    if (act && !act[vinst[v]]) return;  // instance not iterating
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    if (gl) {
        int k = ediag[v];
        for (int j = sptr[k]; j < sptr[k + 1]; ++j) {
            int s = src[j];
            int t = s >> 4, a = (s >> 2) & 3;
            const double* h = gl + 12 * (size_t)t + 3 * a;
            a0 += h[0];
            a1 += h[1];
            a2 += h[2];
        }
    }
    if (Xt) {
        double m = mass[v];
        a0 += m * (X[3 * v] - Xt[3 * v]);
        a1 += m * (X[3 * v + 1] - Xt[3 * v + 1]);
        a2 += m * (X[3 * v + 2] - Xt[3 * v + 2]);
    }
    if (cdiag) {
        int cb = cdiag[v];
        if (cb >= 0)
            for (unsigned j = cseg[cb]; j < cseg[cb + 1]; ++j) {
                unsigned e = cval[j];  // constraint*16 + a*nv + a  (nv packed in bits 28..)
                unsigned i = (e & 0x0FFFFFFFu) >> 4, slot = e >> 28;
                const double* h = gb + 12 * (size_t)i + 3 * slot;
                a0 += h[0];
                a1 += h[1];
                a2 += h[2];
            }
    }
    if (dbc && dbc[v]) a0 = a1 = a2 = 0.0;
    if (g) {
        g[3 * v] = a0;
        g[3 * v + 1] = a1;
        g[3 * v + 2] = a2;
    }
    if (rhs) {
        rhs[3 * v] = -a0;
        rhs[3 * v + 1] = -a1;
        rhs[3 * v + 2] = -a2;
    }
}

// ---------------------------------------------------------------------------
// contact blocks: keys, sort, run heads, reduction
// ---------------------------------------------------------------------------
__global__ void k_contact_nv2(long n, const int* __restrict__ nv, unsigned* __restrict__ cnt)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    cnt[i] = (unsigned)(nv[i] * nv[i]);
}

// record value: (slot_row << 28) | (constraint*16 + a*nv + b); slot_row = a
__global__ void k_contact_keys(long n, const int* __restrict__ vid, const int* __restrict__ nv,
                               const unsigned* __restrict__ off, unsigned long long V,
                               unsigned long long* __restrict__ keys, unsigned* __restrict__ vals)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int k = nv[i];
    unsigned o = off[i];
    for (int a = 0; a < k; ++a)
        for (int b = 0; b < k; ++b) {
            keys[o] = (unsigned long long)vid[4 * i + a] * V + (unsigned long long)vid[4 * i + b];
            vals[o] = ((unsigned)a << 28) | (unsigned)(i * 16 + a * k + b);
            ++o;
        }
}

__global__ void k_run_heads(unsigned n, const unsigned long long* __restrict__ keys, unsigned* __restrict__ head)
{
    unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    head[i] = (i < n && (i == 0 || keys[i] != keys[i - 1])) ? 1u : 0u;
}

__global__ void k_contact_pattern(unsigned n, const unsigned long long* __restrict__ keys,
                                  const unsigned* __restrict__ hs, unsigned long long V, unsigned nb,
                                  unsigned* __restrict__ seg,
                                  int* __restrict__ crow, int* __restrict__ ccol, int* __restrict__ cdiag)
{
    unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == 0) seg[nb] = n;
    if (!(i == 0 || keys[i] != keys[i - 1])) return;
    unsigned b = hs[i];
    seg[b] = i;
    int r = (int)(keys[i] / V), c = (int)(keys[i] % V);
    crow[b] = r;
    ccol[b] = c;
    if (r == c) cdiag[r] = (int)b;
}

__global__ void k_rowptr_from_rows(unsigned nb, const int* __restrict__ row, int nV, int* __restrict__ rowptr)
{
    // rowptr[r] = first block with row >= r (rows sorted)
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > nV) return;
    unsigned lo = 0, hi = nb;
    while (lo < hi) {
        unsigned mid = (lo + hi) >> 1;
        if (row[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    rowptr[r] = (int)lo;
}

__global__ void k_contact_values(unsigned nb, const unsigned* __restrict__ seg, const unsigned* __restrict__ vals,
                                 const double* __restrict__ Hb, const int* __restrict__ crow,
                                 const int* __restrict__ vinst, const unsigned char* __restrict__ act,
                                 double* __restrict__ cval)
{
    unsigned b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    if (act && !act[vinst[crow[b]]]) return;  // instance not iterating
    double acc[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) acc[i] = 0.0;
    for (unsigned j = seg[b]; j < seg[b + 1]; ++j) {
        const double* h = Hb + 9 * (size_t)(vals[j] & 0x0FFFFFFFu);
#pragma unroll
        for (int i = 0; i < 9; ++i) acc[i] += h[i];
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) cval[i * (size_t)nb + b] = acc[i];  // component planes
}

// DBC projection (CSR_MATRIX.h:130-141): blocks touching a DBC node -> delta_ij
__global__ void k_project_dbc(long nnzb, const int* __restrict__ row, const int* __restrict__ col,
                              const unsigned char* __restrict__ dbc, int keep_diag_identity, double* __restrict__ val)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnzb) return;
    int r = row[k], c = col[k];
    if (!(dbc[r] || dbc[c])) return;
    double d = (r == c && keep_diag_identity) ? 1.0 : 0.0;
#pragma unroll
    for (int i = 0; i < 9; ++i) val[i * (size_t)nnzb + k] = (i % 4 == 0) ? d : 0.0;
}

// ---------------------------------------------------------------------------
// PCG kernels
// ---------------------------------------------------------------------------
// block-Jacobi: inverse of E_vv + C_vv
__global__ void k_block_jacobi(int nV, const int* __restrict__ ediag, const double* __restrict__ evals, long eld,
                               const int* __restrict__ cdiag, const double* __restrict__ cvals, long cld,
                               const int* __restrict__ vinst, double* __restrict__ Pinv, int* __restrict__ err)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV) return;
    double a[9];
    const long ed = ediag[v];
#pragma unroll
    for (int i = 0; i < 9; ++i) a[i] = evals[i * eld + ed];
    if (cdiag) {
        int c = cdiag[v];
        if (c >= 0)
#pragma unroll
            for (int i = 0; i < 9; ++i) a[i] += cvals[i * cld + c];
    }
    double c0 = a[4] * a[8] - a[5] * a[7], c1 = a[5] * a[6] - a[3] * a[8], c2 = a[3] * a[7] - a[4] * a[6];
    double det = a[0] * c0 + a[1] * c1 + a[2] * c2;
    double* o = Pinv + 9 * (size_t)v;
    if (!(det > 0)) {
        atomicOr(err + vinst[v], 1);
        det = 1.0;
    }
    double id = 1.0 / det;
    o[0] = c0 * id;
    o[3] = c1 * id;
    o[6] = c2 * id;
    o[1] = (a[2] * a[7] - a[1] * a[8]) * id;
    o[4] = (a[0] * a[8] - a[2] * a[6]) * id;
    o[7] = (a[1] * a[6] - a[0] * a[7]) * id;
    o[2] = (a[1] * a[5] - a[2] * a[4]) * id;
    o[5] = (a[2] * a[3] - a[0] * a[5]) * id;
    o[8] = (a[0] * a[4] - a[1] * a[3]) * id;
}

// ---------------------------------------------------------------------------
// Cluster block-Jacobi preconditioner.  Stiff barrier terms couple the
// vertices of a contact pair far more strongly than mass or elasticity do,
// and a 3x3 block-Jacobi leaves those couplings (and the elastic ones) to the
// iteration.  Vertices are grouped by two rounds of mutual heavy-edge
// matching over the off-diagonal blocks, elastic and contact (contact only
// with precond 2), into clusters of at most 4 vertices, never across
// instances; each cluster's (3k)^2 diagonal block of E + C is inverted
// exactly.  Vertex v stores the 3 x 3k rows of its cluster inverse as k 3x3
// blocks (plane b for member b), z_v = sum_b Z_vb r_mb, and the member list
// (ascending, -1 padded) as one int4, so the PCG reads both without a
// dependent load.
// ---------------------------------------------------------------------------
constexpr int CL_MAX = 4;
constexpr int CL_ZS = 9 * CL_MAX;  // doubles of preconditioner rows per vertex

__device__ inline double cblock_norm2(const double* __restrict__ val, long ld, int k)
{
    double w = 0.0;
#pragma unroll
    for (int e = 0; e < 9; ++e) w += val[e * ld + k] * val[e * ld + k];
    return w;
}

// vertices of the instances that solve (act null: all); every cluster lies
// in one instance, so a skipped vertex is never read by a kept one
struct ClMask {
    const int* vinst;
    const unsigned char* act;
    __device__ bool skip(int v) const { return act && !act[vinst[v]]; }
};

// elastic blocks taken into the matching as well (precond 0); rp null: contact blocks only
struct ClElastic {
    const int* rp;
    const int* col;
    const double* val;
    long ld;
};

// The rows of the two matching passes are read by groups of CL_LANES lanes,
// neighbouring lanes taking neighbouring blocks, so that a plane's loads
// share lines (one lane per row: 94 us a pass on the 64x16x16 bar, 800 us on
// 386,561 rows).
constexpr int CL_LANES = 8;

// strongest contact neighbour of every vertex (ties: smaller id); -1 if none
__global__ void k_cl_best(int nV, const int* __restrict__ crp, const int* __restrict__ ccol,
                          const double* __restrict__ cval, long cld, ClElastic el, ClMask cm,
                          int* __restrict__ best)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int v = (int)(t / CL_LANES), lane = (int)(t % CL_LANES);
    if (v >= nV || cm.skip(v)) return;  // uniform over the group
    int b = -1;
    double bw = 0.0;
    auto consider = [&](int u, double w) {
        if (u != v && (w > bw || (w == bw && b >= 0 && u < b))) {
            bw = w;
            b = u;
        }
    };
    if (crp)
        for (int k = crp[v] + lane; k < crp[v + 1]; k += CL_LANES) consider(ccol[k], cblock_norm2(cval, cld, k));
    if (el.rp)
        for (int k = el.rp[v] + lane; k < el.rp[v + 1]; k += CL_LANES)
            consider(el.col[k], cblock_norm2(el.val, el.ld, k));
#pragma unroll
    for (int o = CL_LANES / 2; o > 0; o >>= 1) {
        const int u = __shfl_xor(b, o, CL_LANES);
        const double w = __shfl_xor(bw, o, CL_LANES);
        if (u >= 0 && (w > bw || (w == bw && (b < 0 || u < b)))) {
            bw = w;
            b = u;
        }
    }
    if (lane == 0) best[v] = b;
}

__global__ void k_cl_pair(int nV, const int* __restrict__ best, ClMask cm, int* __restrict__ root,
                          int* __restrict__ size)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV || cm.skip(v)) return;
    const int b = best[v];
    const bool pair = b >= 0 && best[b] == v;
    root[v] = pair ? min(v, b) : v;
    size[v] = pair ? 2 : 1;  // meaningful at roots
}

// second matching pass: strongest neighbouring cluster of every cluster (max
// block norm over member-to-member blocks, contact and, with precond 0,
// elastic), packed (float weight, -root) so that a 64-bit max picks the
// heaviest, then the lowest root
__global__ void k_cl_best2(int nV, const int* __restrict__ crp, const int* __restrict__ ccol,
                           const double* __restrict__ cval, long cld, const int* __restrict__ root,
                           const int* __restrict__ size, ClElastic el, ClMask cm,
                           unsigned long long* __restrict__ pack)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int v = (int)(t / CL_LANES), lane = (int)(t % CL_LANES);
    if (v >= nV || (!crp && !el.rp) || cm.skip(v)) return;  // uniform over the group
    const int r = root[v];
    unsigned long long bestp = 0;
    auto consider = [&](int u, double w) {
        const int ru = root[u];
        if (ru == r || size[r] + size[ru] > CL_MAX) return;
        const float wf = (float)w;
        const unsigned long long p =
            ((unsigned long long)__float_as_uint(wf) << 32) | (unsigned long long)(0xFFFFFFFFu - (unsigned)ru);
        if (p > bestp) bestp = p;
    };
    if (crp)
        for (int k = crp[v] + lane; k < crp[v + 1]; k += CL_LANES) consider(ccol[k], cblock_norm2(cval, cld, k));
    if (el.rp)
        for (int k = el.rp[v] + lane; k < el.rp[v + 1]; k += CL_LANES)
            consider(el.col[k], cblock_norm2(el.val, el.ld, k));
#pragma unroll
    for (int o = CL_LANES / 2; o > 0; o >>= 1) {
        const unsigned long long p = __shfl_xor(bestp, o, CL_LANES);
        bestp = p > bestp ? p : bestp;
    }
    if (lane == 0 && bestp) atomicMax(pack + r, bestp);
}

__global__ void k_cl_merge(int nV, int* __restrict__ root, const unsigned long long* __restrict__ pack,
                           int* __restrict__ size, ClMask cm, int* __restrict__ root2)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV || cm.skip(v)) return;
    const int r = root[v];
    int nr = r;
    const unsigned long long p = pack[r];
    if (p) {
        const int b = (int)(0xFFFFFFFFu - (unsigned)(p & 0xFFFFFFFFull));
        const unsigned long long q = pack[b];
        if (q && (int)(0xFFFFFFFFu - (unsigned)(q & 0xFFFFFFFFull)) == r) nr = min(r, b);
    }
    root2[v] = nr;
}

__global__ void k_cl_members(int nV, const int* __restrict__ root, ClMask cm, int* __restrict__ cnt,
                             int* __restrict__ mem)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV || cm.skip(v)) return;
    const int r = root[v];
    const int slot = atomicAdd(cnt + r, 1);
    if (slot < CL_MAX) mem[CL_MAX * r + slot] = v;
}

// members of each cluster in ascending order
__global__ void k_cl_sort(int nV, const int* __restrict__ root, const int* __restrict__ cnt, ClMask cm,
                          int* __restrict__ mem)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nV || cm.skip(v)) return;
    const int r = root[v];
    const int k = min(cnt[r], CL_MAX);
    if (v == r) {
        int* m = mem + CL_MAX * r;
        for (int i = 1; i < k; ++i)
            for (int j = i; j > 0 && m[j - 1] > m[j]; --j) {
                const int t = m[j - 1];
                m[j - 1] = m[j];
                m[j] = t;
            }
    }
}

// locate block (a, b) in a BSR row; returns -1 when absent (8 columns are
// read together)
__device__ inline int bsr_find(const int* __restrict__ rp, const int* __restrict__ col, int a, int b)
{
    const int e = rp[a + 1];
    int f = -1;
    for (int k = rp[a]; k < e && f < 0; k += 8) {
        int c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = col[min(k + u, e - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k + u < e && c[u] == b) f = k + u;
    }
    return f;
}

// Gathers a cluster's (3k)^2 block of E + C, factors it (Cholesky), inverts
// it and scatters the member rows to Z, by 16 lanes per vertex (the group of
// the cluster's root works): lane 4a + b gathers the 3x3 block of members a
// and b, lane i holds row i of the factorization, lane c forms column c of the
// inverse.  The factor is padded to order 12 with the identity, so every loop
// is unrolled and the rows stay in registers; each entry is formed by the same
// operations in the same order as a sequential Cholesky.  One thread per
// cluster with its matrices in memory took 157 us on 81 rows and 370 us on
// 18,785 (a chain of dependent loads).  Singletons keep the 3x3 inverse of the
// block-Jacobi preconditioner (same arithmetic).
constexpr int CL_N = 3 * CL_MAX;
__global__ void __launch_bounds__(256) k_cl_build(
    int nV, const int* __restrict__ root, const int* __restrict__ cnt, const int* __restrict__ mem,
    const int* __restrict__ ediag, const int* __restrict__ erp, const int* __restrict__ ecol,
    const double* __restrict__ evals, long eld, const int* __restrict__ cdiag, const int* __restrict__ crp,
    const int* __restrict__ ccol, const double* __restrict__ cvals, long cld, const int* __restrict__ vinst, ClMask cmask,
    double* __restrict__ Z, int4* __restrict__ cm4, int* __restrict__ err)
{
    __shared__ double sh[16][CL_N][CL_N + 1];
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int r = (int)(t >> 4), g = (int)(t & 15);
    double(*M)[CL_N + 1] = sh[threadIdx.x >> 4];
    // uniform over the group of 16 lanes
    const bool work = r < nV && !cmask.skip(r) && root[r] == r;
    const int k = work ? min(cnt[r], CL_MAX) : 0;
    const int* m = mem + CL_MAX * (size_t)min(r, nV - 1);
    int mm[CL_MAX];
#pragma unroll
    for (int a = 0; a < CL_MAX; ++a) mm[a] = a < k ? m[a] : -1;
    if (work && g < k) cm4[m[g]] = make_int4(mm[0], mm[1], mm[2], mm[3]);
    if (k == 1 && g == 0) {
        double a[9];
        const long ed = ediag[r];
#pragma unroll
        for (int i = 0; i < 9; ++i) a[i] = evals[i * eld + ed];
        if (cdiag) {
            const int c = cdiag[r];
            if (c >= 0)
#pragma unroll
                for (int i = 0; i < 9; ++i) a[i] += cvals[i * cld + c];
        }
        double c0 = a[4] * a[8] - a[5] * a[7], c1 = a[5] * a[6] - a[3] * a[8], c2 = a[3] * a[7] - a[4] * a[6];
        double det = a[0] * c0 + a[1] * c1 + a[2] * c2;
        double* o = Z + 9 * (size_t)r;  // plane 0
        if (!(det > 0)) {
            atomicOr(err + vinst[r], 1);
            det = 1.0;
        }
        double id = 1.0 / det;
        o[0] = c0 * id;
        o[3] = c1 * id;
        o[6] = c2 * id;
        o[1] = (a[2] * a[7] - a[1] * a[8]) * id;
        o[4] = (a[0] * a[8] - a[2] * a[6]) * id;
        o[7] = (a[1] * a[6] - a[0] * a[7]) * id;
        o[2] = (a[1] * a[5] - a[2] * a[4]) * id;
        o[5] = (a[2] * a[3] - a[0] * a[5]) * id;
        o[8] = (a[0] * a[4] - a[1] * a[3]) * id;
    }
    const bool big = k > 1;
    // ---- gather
    {
        const int a = g >> 2, b = g & 3;
        double blk[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) blk[i] = (a == b && i % 4 == 0 && a >= k) ? 1.0 : 0.0;
        if (big && a < k && b < k) {
            const int ke = bsr_find(erp, ecol, m[a], m[b]);
            if (ke >= 0)
#pragma unroll
                for (int i = 0; i < 9; ++i) blk[i] += evals[i * eld + ke];
            if (crp) {
                const int kc = bsr_find(crp, ccol, m[a], m[b]);
                if (kc >= 0)
#pragma unroll
                    for (int i = 0; i < 9; ++i) blk[i] += cvals[i * cld + kc];
            }
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) M[3 * a + i][3 * b + j] = blk[3 * i + j];
    }
    __syncthreads();
    // ---- row i of the lower triangle, symmetrised (the assembled blocks are
    // symmetric up to rounding), factored column by column
    const int row = min(g, CL_N - 1);
    double L[CL_N];
#pragma unroll
    for (int j = 0; j < CL_N; ++j) L[j] = j == row ? M[row][j] : 0.5 * (M[row][j] + M[j][row]);
    bool ok = true;
#pragma unroll
    for (int q = 0; q < CL_N; ++q) {
        const double d = __shfl(L[q], q, 16);
        ok = ok && d > 0;
        const double lqq = sqrt(d);
        L[q] = row == q ? lqq : L[q] / lqq;
#pragma unroll
        for (int j = q + 1; j < CL_N; ++j) L[j] -= L[q] * __shfl(L[q], j, 16);
    }
    __syncthreads();  // every lane has read M
    if (g < CL_N)
#pragma unroll
        for (int j = 0; j < CL_N; ++j)
            if (j <= g) M[g][j] = L[j];
    __syncthreads();
    if (!big) return;
    // ---- column c of the inverse: L y = e_c, L^T x = y
    const int c = row;
    double y[CL_N];
#pragma unroll
    for (int i = 0; i < CL_N; ++i) {
        double s = i == c ? 1.0 : 0.0;
#pragma unroll
        for (int q = 0; q < i; ++q) s -= M[i][q] * y[q];
        y[i] = s / M[i][i];
    }
#pragma unroll
    for (int i = CL_N - 1; i >= 0; --i) {
        double s = y[i];
#pragma unroll
        for (int q = i + 1; q < CL_N; ++q) s -= M[q][i] * y[q];
        y[i] = s / M[i][i];
    }
    if (!ok) {
        if (g == 0) atomicOr(err + vinst[r], 1);
#pragma unroll
        for (int i = 0; i < CL_N; ++i) y[i] = i == c ? 1.0 : 0.0;
    }
    // ---- member a's rows, as k 3x3 blocks: block (a, b) in plane b at row m[a]
    if (g < 3 * k) {
        const int b = g / 3, j = g % 3;
#pragma unroll
        for (int a = 0; a < CL_MAX; ++a)
            if (a < k) {
                double* o = Z + 9 * ((size_t)b * nV + mm[a]);
#pragma unroll
                for (int i = 0; i < 3; ++i) o[3 * i + j] = y[3 * a + i];
            }
    }
}

// z_v = Z_v r_members (members' r given by rfun).  Z holds CL_MAX planes of
// 9 nV doubles: the 3x3 block of vertex v for its cluster's b-th member is
// at plane b, row v, so singletons (most vertices) read plane 0 only and a
// wavefront's reads of a plane are contiguous.
template <class RF>
__device__ inline void cl_apply(int4 cm, const double* __restrict__ Z, int nV, int v, const double* own, RF&& rfun,
                                double* zv)
{
    const double* o = Z + 9 * (size_t)v;
    if (cm.y < 0) {  // singleton: the 3x3 inverse of the diagonal block
#pragma unroll
        for (int i = 0; i < 3; ++i) zv[i] = o[3 * i] * own[0] + o[3 * i + 1] * own[1] + o[3 * i + 2] * own[2];
        return;
    }
    const int mb[CL_MAX] = {cm.x, cm.y, cm.z, cm.w};
    zv[0] = zv[1] = zv[2] = 0.0;
#pragma unroll
    for (int b = 0; b < CL_MAX; ++b) {
        if (mb[b] < 0) break;
        double rb[3];
        rfun(mb[b], rb);
        const double* ob = o + 9 * (size_t)b * nV;
#pragma unroll
        for (int i = 0; i < 3; ++i) zv[i] += ob[3 * i] * rb[0] + ob[3 * i + 1] * rb[1] + ob[3 * i + 2] * rb[2];
    }
}

// ---------------------------------------------------------------------------
// Block-Jacobi PCG as two kernels per iteration, enqueued in chunks with no
// host synchronisation inside a chunk (smaller systems run as one kernel,
// k_pcg_team below).
//  * k_pcg_spmv(it): every block re-reduces the previous update's partials
//    (r.z, r.r) in a fixed order, decides convergence identically, forms
//    p_it = z + beta p_(it-1) on the fly and computes q = A p_it with a group
//    of PCG_G lanes per block row (xor-butterfly row reduction), plus
//    partial p.q.
//  * k_pcg_update(it): alpha = r.z / p.q; x += alpha p; r -= alpha q; z = P r;
//    partials of the new r.z and r.r.
// p and the r.z / r.r partials ping-pong on the iteration parity.  When the
// residual test holds (or on breakdown), the deciding kernel sets a flag and
// every later kernel returns at once, so the host may enqueue past the end.
// ---------------------------------------------------------------------------
struct PcgArgs {
    int nV;
    const int* erp;
    const int* ecol;
    const double* eval;  // 9 component planes of eld blocks
    const int* crp;      // null when there are no contact blocks
    const int* ccol;
    const double* cval;  // 9 component planes of cld blocks
    long eld, cld;
    const double* b;
    const double* Z;      // preconditioner rows: CL_MAX planes of 9 nV doubles (cl_apply)
    const int4* cm4;      // per vertex: its cluster's members, ascending, -1 padded
    double* x;
    double* r;        // 2 x 3V: the update of iteration it reads half it&1, writes the other
    double* z;
    double* pbuf;     // 2 x 3V
    double* q;
    double* part_pq;  // nbA
    double* part_bx;  // nbA: b.x of the warm-start pass
    const unsigned char* warm;  // per instance: start from gamma x (x holds the previous direction); null = none
    double* part_rz;  // 2 x nbB
    double* part_rr;  // 2 x nbB
    int nbA, nbB;
    // launch tables: one int4 {first row, end row, instance, block id} per
    // launched block, SpMV blocks of PCG_ROWS rows (atab) and update blocks of
    // 64 rows (btab), each aligned to its instance's first row.  Only the
    // blocks of instances still iterating are launched; partials are indexed
    // by the block id, so an instance's partial range [apbeg, bpbeg) is the
    // same whatever else is launched.
    const int4 *atab, *btab;
    const int *aoff, *boff;  // per launched block: iterations its instance did in earlier calls
    int ident;               // one instance, all blocks launched: entries follow from blockIdx (no table load)
    int nbl_upd;             // update blocks launched (upd_waves per workgroup)
    const int *apbeg, *bpbeg;
    const unsigned char* solve;  // per instance: 0 not solving, 1 new solve, 2 continued from an earlier call
    int* flag;        // per instance: 0 running, 1 converged, 2 breakdown, 3 not solving, 4 maxit reached
    double* scal;     // per instance, 3 each: |b|^2, final |r|^2, iterations
    double rtol2;
    int maxit;
    // one instance with many blocks: the sums of the partials are formed once
    // per kernel boundary by k_pcg_red_spmv / k_pcg_red_upd (r.z, r.r, the
    // previous r.z or |b|^2; p.q, r.z) instead of by every block (null)
    double* red;
    // coarse level (one instance): partials of r_c . e_c, cnsb per parity,
    // added to r.z wherever it is formed (null: none)
    const double* cpart;
    int cnsb;
};

constexpr int PCG_ROW_THREADS = 256;         // row threads of a SpMV block (4 wavefronts), 256 / G rows
constexpr int PCG_PREREDUCE_BLOCKS = 1024;   // update blocks of one instance from which partials are pre-reduced
constexpr int PCG_UPD_BLOCK = 64;            // rows of an update block: one wavefront, reductions need no barrier
constexpr int PCG_UPD_WAVES_MAX = 8;         // update blocks per workgroup (independent wavefronts), at most
// SpMV launch shapes: G lanes per block row, scalars in wavefront 0 (before
// its rows) or in a fifth wavefront of their own
struct SpmvShape {
    int g;
    bool sw;
};
constexpr SpmvShape SPMV_SHAPES[] = {{4, false}, {8, false}, {16, false}, {32, false},
                                     {4, true},  {8, true},  {16, true},  {32, true}};
inline int spmv_rows(int g) { return PCG_ROW_THREADS / g; }

// Launch-table entry of this block: {first row, end row, instance, block id}.
// A one-instance launch derives it from blockIdx, saving a dependent load.
template <int ROWS>
__device__ inline int4 launch_entry(const PcgArgs& A, const int4* __restrict__ tab, int blk)
{
    if (A.ident) {
        const int lo = blk * ROWS;
        return make_int4(lo, min(lo + ROWS, A.nV), 0, blk);
    }
    return tab[blk];
}
template <int ROWS>
__device__ inline int4 launch_entry(const PcgArgs& A, const int4* __restrict__ tab)
{
    return launch_entry<ROWS>(A, tab, (int)blockIdx.x);
}
__device__ inline int launch_off(const PcgArgs& A, const int* __restrict__ off, int blk)
{
    return A.ident ? A.ident - 1 : off[blk];
}
__device__ inline int launch_off(const PcgArgs& A, const int* __restrict__ off)
{
    return launch_off(A, off, (int)blockIdx.x);
}

// Sum over a wavefront by a fixed xor butterfly (every lane gets the total).
__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sum of n partials by one wavefront in a fixed order.  The loads of a chunk
// of NL per lane are issued together (independent), then added in order, so
// the latency is paid once per 64 NL partials rather than once per 64.
template <int NL = 16>
__device__ inline double wave_sum_partials(const double* __restrict__ part, int n)
{
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    for (int base = 0; base < n; base += 64 * NL) {
        double v[NL];
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            const int i = base + lane + 64 * k;
            v[k] = i < n ? part[i] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < NL; ++k) acc += v[k];
    }
    return wave_sum(acc);
}

// Three sums of n partials each, every load issued before any add (one
// memory round trip for up to 512 partials per array); each sum is formed in
// the order wave_sum_partials uses, so the results are the same.
__device__ inline void wave_sum_partials3(const double* __restrict__ p0, const double* __restrict__ p1,
                                          const double* __restrict__ p2, int n, double& s0, double& s1,
                                          double& s2)
{
    const int lane = threadIdx.x & 63;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (int base = 0; base < n; base += 64 * 8) {
        double v0[8], v1[8], v2[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i = base + lane + 64 * k;
            const bool in = i < n;
            v0[k] = in ? p0[i] : 0.0;
            v1[k] = in ? p1[i] : 0.0;
            v2[k] = in ? p2[i] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            a0 += v0[k];
            a1 += v1[k];
            a2 += v2[k];
        }
    }
    s0 = wave_sum(a0);
    s1 = wave_sum(a1);
    s2 = wave_sum(a2);
}

// Two sums of partials (na and nb of them) with the first NA and NB loads
// per lane of both issued before any add; the per-lane order of the adds is
// that of wave_sum_partials, so the sums are the same.
template <int NA, int NB>
__device__ inline void wave_sum_partials2(const double* __restrict__ pa, int na, const double* __restrict__ pb,
                                          int nb, double& sa, double& sb)
{
    const int lane = threadIdx.x & 63;
    double va[NA], vb[NB];
#pragma unroll
    for (int k = 0; k < NA; ++k) va[k] = lane + 64 * k < na ? pa[lane + 64 * k] : 0.0;
#pragma unroll
    for (int k = 0; k < NB; ++k) vb[k] = lane + 64 * k < nb ? pb[lane + 64 * k] : 0.0;
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int k = 0; k < NA; ++k) a += va[k];
#pragma unroll
    for (int k = 0; k < NB; ++k) b += vb[k];
    for (int i = lane + 64 * NA; i < na; i += 64) a += pa[i];
    for (int i = lane + 64 * NB; i < nb; i += 64) b += pb[i];
    sa = wave_sum(a);
    sb = wave_sum(b);
}

// y += A_row z (and w += A_row po when po is given) over this lane's blocks of
// row v: the row's elastic blocks followed by its contact blocks, lanes of
// a group taking slots lane, lane + G, ...  Rows of at most G blocks
// (most of them) take one slot per lane, so every load of a lane is issued at
// once.  Values are 9 component planes of ld doubles: the lanes of a group
// read consecutive addresses.
template <int G>
__device__ inline void row_spmv(int lane, int e0, int ne, int c0, int nc, const PcgArgs& A,
                                const double* __restrict__ z, const double* __restrict__ po, double* y, double* w)
{
    for (int j = lane; j < ne + nc; j += G) {
        const bool el = j < ne;
        const double* __restrict__ val = el ? A.eval : A.cval;
        const long ld = el ? A.eld : A.cld;
        const int k = el ? e0 + j : c0 + (j - ne);
        const int col = el ? A.ecol[k] : A.ccol[k];
        const double bk[9] = {val[k], val[ld + k], val[2 * ld + k], val[3 * ld + k], val[4 * ld + k],
                              val[5 * ld + k], val[6 * ld + k], val[7 * ld + k], val[8 * ld + k]};
        const size_t c = 3 * (size_t)col;
        const double x0 = z[c], x1 = z[c + 1], x2 = z[c + 2];
        y[0] += bk[0] * x0 + bk[1] * x1 + bk[2] * x2;
        y[1] += bk[3] * x0 + bk[4] * x1 + bk[5] * x2;
        y[2] += bk[6] * x0 + bk[7] * x1 + bk[8] * x2;
        if (po) {
            const double p0 = po[c], p1 = po[c + 1], p2 = po[c + 2];
            w[0] += bk[0] * p0 + bk[1] * p1 + bk[2] * p2;
            w[1] += bk[3] * p0 + bk[4] * p1 + bk[5] * p2;
            w[2] += bk[6] * p0 + bk[7] * p1 + bk[8] * p2;
        }
    }
}

// row extents of row v in both block sets
__device__ inline void row_extents(const PcgArgs& A, int v, int& e0, int& ne, int& c0, int& nc)
{
    e0 = A.erp[v];
    ne = A.erp[v + 1] - e0;
    c0 = A.crp ? A.crp[v] : 0;
    nc = A.crp ? A.crp[v + 1] - c0 : 0;
}

template <int G>
__device__ inline double row_butterfly(double* y, int lane)
{
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        y[0] += __shfl_xor(y[0], o, G);
        y[1] += __shfl_xor(y[1], o, G);
        y[2] += __shfl_xor(y[2], o, G);
    }
    // select by value (an index into y would put the array in scratch memory)
    const double y0 = y[0], y1 = y[1], y2 = y[2];
    double r = y2;
    r = lane == 1 ? y1 : r;
    r = lane == 0 ? y0 : r;
    return r;
}

// sum of one double per thread of the row threads -> one partial per block
__device__ inline double block_row_sum(double v, double* wsum)
{
    v = wave_sum(v);
    if (threadIdx.x < PCG_ROW_THREADS && (threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    double a = 0.0;
#pragma unroll
    for (int w2 = 0; w2 < PCG_ROW_THREADS / 64; ++w2) a += wsum[w2];
    return a;
}

// x0 = gamma x_prev (gamma = b.x / x.Ax, the A-norm-closest multiple of the
// previous direction) for warm instances, else 0; r0 = b - gamma A x_prev;
// z0 = P r0; partials of r.z, r.r and b.b (the last in the second half of
// the r.r partials, read by the first SpMV)
__global__ void __launch_bounds__(PCG_UPD_BLOCK) k_pcg_init(PcgArgs A)
{
    const int4 t = launch_entry<PCG_UPD_BLOCK>(A, A.btab);
    const int inst = t.z, bid = t.w;
    if (A.flag[inst] != 0 || (A.solve && A.solve[inst] != 1)) return;  // not solving, or continued
    const int v = t.x + threadIdx.x;
    double gamma = 0.0;
    if (A.warm && A.warm[inst]) {
        const int ab = A.apbeg[inst], na = A.apbeg[inst + 1] - ab;
        const double xq = wave_sum_partials<32>(A.part_pq + ab, na);
        const double bx = wave_sum_partials<32>(A.part_bx + ab, na);
        gamma = xq > 0.0 ? bx / xq : 0.0;
    }
    const bool w = gamma != 0.0;
    auto res = [&](int u, double* o) {
#pragma unroll
        for (int i = 0; i < 3; ++i) o[i] = w ? A.b[3 * u + i] - gamma * A.q[3 * u + i] : A.b[3 * u + i];
    };
    double drz = 0.0, drr = 0.0, dbb = 0.0;
    if (v < t.y) {
        double rv[3], zv[3];
        res(v, rv);
        cl_apply(A.cm4[v], A.Z, A.nV, v, rv, res, zv);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double bi = A.b[3 * v + i];
            A.x[3 * v + i] = w ? gamma * A.x[3 * v + i] : 0.0;
            A.r[3 * v + i] = rv[i];
            A.z[3 * v + i] = zv[i];
            A.pbuf[3 * ((size_t)A.nV + v) + i] = 0.0;  // p before the first iteration
            drz += rv[i] * zv[i];
            drr += rv[i] * rv[i];
            dbb += bi * bi;
        }
    }
    drz = wave_sum(drz);
    drr = wave_sum(drr);
    dbb = wave_sum(dbb);
    if (threadIdx.x == 0) {
        A.part_rz[bid] = drz;
        A.part_rr[bid] = drr;
        A.part_rr[A.nbB + bid] = dbb;
    }
}

// warm start: q = A x for the instances that start from their previous
// direction, with per-block partials of x.q and b.x
template <int G>
__global__ void __launch_bounds__(PCG_ROW_THREADS) k_pcg_warm(PcgArgs A)
{
    __shared__ double wsum[2][PCG_ROW_THREADS / 64];
    const int4 t = launch_entry<PCG_ROW_THREADS / G>(A, A.atab);
    const int inst = t.z;
    const bool on = A.warm[inst] && A.flag[inst] == 0;  // uniform over the block
    const int lane = threadIdx.x & (G - 1);
    const int v = t.x + threadIdx.x / G;
    const bool row = on && threadIdx.x < PCG_ROW_THREADS && v < t.y;
    double y[3] = {0.0, 0.0, 0.0}, w[3] = {0.0, 0.0, 0.0};
    double dxq = 0.0, dbx = 0.0;
    if (row) {
        int e0, ne, c0, nc;
        row_extents(A, v, e0, ne, c0, nc);
        row_spmv<G>(lane, e0, ne, c0, nc, A, A.x, nullptr, y, w);
        const double yl = row_butterfly<G>(y, lane);
        if (lane < 3) {
            const size_t i = 3 * (size_t)v + lane;
            const double xi = A.x[i];
            A.q[i] = yl;
            dxq = xi * yl;
            dbx = A.b[i] * xi;
        }
    }
    dxq = wave_sum(dxq);
    dbx = wave_sum(dbx);
    if (threadIdx.x < PCG_ROW_THREADS && (threadIdx.x & 63) == 0) {
        wsum[0][threadIdx.x >> 6] = dxq;
        wsum[1][threadIdx.x >> 6] = dbx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, c = 0.0;
#pragma unroll
        for (int w2 = 0; w2 < PCG_ROW_THREADS / 64; ++w2) {
            a += wsum[0][w2];
            c += wsum[1][w2];
        }
        A.part_pq[t.w] = a;
        A.part_bx[t.w] = c;
    }
}

// SpMV step of iteration it.  The scalar wavefront re-reduces the instance's
// partials of the previous update and decides convergence while the row
// wavefronts stream their blocks; p_it = z + beta p_(it-1) is never read:
// the rows accumulate A z and A p_(it-1) separately and combine them once
// beta is known, q = A z + beta A p_(it-1).
template <int G, bool SW>
__global__ void __launch_bounds__(PCG_ROW_THREADS + (SW ? 64 : 0)) k_pcg_spmv(PcgArgs A, int it_call)
{
    __shared__ double sbeta;
    __shared__ double wsum[PCG_ROW_THREADS / 64];
    __shared__ int sflag;
    const int it = it_call + launch_off(A, A.aoff);  // the instance's own iteration
    const int par = it & 1;
    const int4 t = launch_entry<PCG_ROW_THREADS / G>(A, A.atab);
    const int inst = t.z, bid = t.w;
    const double* po = it > 0 ? A.pbuf + (size_t)(par ^ 1) * 3 * A.nV : nullptr;
    double y[3] = {0.0, 0.0, 0.0}, w[3] = {0.0, 0.0, 0.0};
    double zo = 0.0, poo = 0.0;
    const int lane = threadIdx.x & (G - 1);
    const int v = t.x + threadIdx.x / G;
    bool row = false;
    auto scalars = [&]() {
        const int f = *(volatile int*)(A.flag + inst);
        const int pb = A.bpbeg[inst], np = A.bpbeg[inst + 1] - pb;
        // r.z and r.r of this iteration, and r.z of the previous one (|b|^2 at it = 0)
        double rz, rr, third;
        if (A.red) {
            rz = A.red[0];
            rr = A.red[1];
            third = A.red[2];
        } else {
            wave_sum_partials3(A.part_rz + par * A.nbB + pb, A.part_rr + par * A.nbB + pb,
                               it > 0 ? A.part_rz + (par ^ 1) * A.nbB + pb : A.part_rr + A.nbB + pb, np, rz, rr,
                               third);
        }
        if (A.cpart) {  // r . (z1 + P e_c) = r . z1 + r_c . e_c
            rz += wave_sum_partials<8>(A.cpart + par * A.cnsb, A.cnsb);
            if (it > 0) third += wave_sum_partials<8>(A.cpart + (par ^ 1) * A.cnsb, A.cnsb);
        }
        const double rzo = it > 0 ? third : 1.0;
        const double bbp = it == 0 ? third : 0.0;
        if ((threadIdx.x & 63) == 0) {
            double* sci = A.scal + 3 * inst;
            const double bb = it == 0 ? bbp : sci[0];
            int stop = f != 0 ? 2 : 0;
            const bool conv = !(bb > 0.0) || (it > 0 && rr <= A.rtol2 * bb);
            if (!stop && (conv || it >= A.maxit)) {
                stop = 1;
                if (bid == A.apbeg[inst]) {
                    A.flag[inst] = conv ? 1 : 4;  // 4: the iteration limit ended the solve
                    sci[0] = bb;
                    sci[1] = rr;
                    sci[2] = (double)it;
                }
            }
            if (!stop && it == 0 && bid == A.apbeg[inst]) sci[0] = bb;
            sflag = stop;
            sbeta = it > 0 ? rz / rzo : 0.0;
        }
    };
    const bool scalar_wave = SW ? threadIdx.x >= PCG_ROW_THREADS : threadIdx.x < 64;
    if (!SW && scalar_wave) scalars();
    if (threadIdx.x < PCG_ROW_THREADS && v < t.y) {
        // the flag is loaded with the row extents; a stopped instance skips its blocks
        const int f = *(volatile int*)(A.flag + inst);
        int e0, ne, c0, nc;
        row_extents(A, v, e0, ne, c0, nc);
        if (lane < 3) {
            zo = A.z[3 * v + lane];
            poo = po ? po[3 * v + lane] : 0.0;
        }
        row = f == 0;
        if (row) row_spmv<G>(lane, e0, ne, c0, nc, A, A.z, po, y, w);
    }
    if (SW && scalar_wave) scalars();
    __syncthreads();
    if (sflag != 0) return;  // block-uniform
    const double beta = sbeta;
    double dpq = 0.0;
    if (row) {
#pragma unroll
        for (int d = 0; d < 3; ++d) y[d] += beta * w[d];
        const double yl = row_butterfly<G>(y, lane);
        if (lane < 3) {
            const size_t i = 3 * (size_t)v + lane;
            const double pv = po ? zo + beta * poo : zo;
            A.pbuf[(size_t)par * 3 * A.nV + i] = pv;
            A.q[i] = yl;
            dpq = pv * yl;
        }
    }
    const double a = block_row_sum(dpq, wsum);
    if (threadIdx.x == 0) A.part_pq[bid] = a;
}

// Sums of n partials by one workgroup of PCG_RED threads in a fixed order:
// thread t adds i = t, t + PCG_RED, ... (loads issued PCG_RED_NL at a time),
// then the workgroup's sums are added in thread order.
constexpr int PCG_RED = 256;
constexpr int PCG_RED_NL = 8;

template <int K>
__device__ inline void block_sums_partials(const double* const* __restrict__ p, int n, double* out)
{
    __shared__ double sh[K][PCG_RED];
    double acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0;
    for (int base = 0; base < n; base += PCG_RED * PCG_RED_NL) {
        double v[K][PCG_RED_NL];
#pragma unroll
        for (int j = 0; j < PCG_RED_NL; ++j) {
            const int i = base + (int)threadIdx.x + PCG_RED * j;
#pragma unroll
            for (int k = 0; k < K; ++k) v[k][j] = i < n ? p[k][i] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < PCG_RED_NL; ++j)
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] += v[k][j];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) sh[k][threadIdx.x] = acc[k];
    __syncthreads();
    if (threadIdx.x < K) {
        double a = 0.0;
        for (int t = 0; t < PCG_RED; ++t) a += sh[threadIdx.x][t];
        out[threadIdx.x] = a;
    }
}

// the sums the SpMV of iteration it needs (one instance spanning the launch)
__global__ void __launch_bounds__(PCG_RED) k_pcg_red_spmv(PcgArgs A, int it_call)
{
    const int it = it_call + A.ident - 1;
    const int par = it & 1;
    const int pb = A.bpbeg[0], np = A.bpbeg[1] - pb;
    const double* p[3] = {A.part_rz + par * A.nbB + pb, A.part_rr + par * A.nbB + pb,
                          it > 0 ? A.part_rz + (par ^ 1) * A.nbB + pb : A.part_rr + A.nbB + pb};
    block_sums_partials<3>(p, np, A.red);
}

// the sums the update of iteration it needs
__global__ void __launch_bounds__(PCG_RED) k_pcg_red_upd(PcgArgs A, int it_call)
{
    const int it = it_call + A.ident - 1;
    const int par = it & 1;
    const int pb = A.bpbeg[0];
    __shared__ double o[2];
    const double* pa[1] = {A.part_pq + A.apbeg[0]};
    const double* pr[1] = {A.part_rz + par * A.nbB + pb};
    block_sums_partials<1>(pa, A.apbeg[1] - A.apbeg[0], o);
    __syncthreads();
    block_sums_partials<1>(pr, A.bpbeg[1] - pb, o + 1);
    __syncthreads();
    if (threadIdx.x == 0) {
        A.red[3] = o[0];
        A.red[4] = o[1];
    }
}

// Update step of iteration it: alpha = r.z / p.q; x += alpha p; r -= alpha q;
// z = P r (cluster members' residuals recomputed from the unwritten half of
// r); partials of the new r.z and r.r.  Every load that does not depend on
// alpha, the cluster's member list and the preconditioner rows included, is
// issued before the partials are reduced.
__global__ void __launch_bounds__(PCG_UPD_BLOCK * PCG_UPD_WAVES_MAX) k_pcg_update(PcgArgs A, int it_call)
{
    // each wavefront is one update block of 64 rows, independent of the
    // others in its workgroup
    const int blk = blockIdx.x * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6);
    if (blk >= A.nbl_upd) return;  // uniform over the wavefront
    const int lane = threadIdx.x & 63;
    const int it = it_call + launch_off(A, A.boff, blk);  // the instance's own iteration
    const int4 t = launch_entry<PCG_UPD_BLOCK>(A, A.btab, blk);
    const int inst = t.z, bid = t.w;
    const int par = it & 1;
    const double* p = A.pbuf + (size_t)par * 3 * A.nV;
    const double* r_in = A.r + (size_t)par * 3 * A.nV;  // not written by this kernel: members read it safely
    double* r_out = A.r + (size_t)(par ^ 1) * 3 * A.nV;
    const int v = t.x + lane;
    const bool own = v < t.y;
    const int vc = own ? v : t.x;
    const int f = *(volatile int*)(A.flag + inst);
    double xv[3], pv[3], rv[3], qv[3], o0[9];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        xv[i] = A.x[3 * vc + i];
        pv[i] = p[3 * vc + i];
        rv[i] = r_in[3 * vc + i];
        qv[i] = A.q[3 * vc + i];
    }
    const int4 cm = A.cm4[vc];
    const double* o = A.Z + 9 * (size_t)vc;  // plane 0
#pragma unroll
    for (int i = 0; i < 9; ++i) o0[i] = o[i];
    // the partials are read in the same round trip as the flag and the rows
    // (a stopped instance's sums are formed and dropped)
    const int pb = A.bpbeg[inst];
    double pq, rz;
    if (A.red) {
        pq = A.red[3];
        rz = A.red[4];
    } else {
        wave_sum_partials2<8, 4>(A.part_pq + A.apbeg[inst], A.apbeg[inst + 1] - A.apbeg[inst],
                                  A.part_rz + par * A.nbB + pb, A.bpbeg[inst + 1] - pb, pq, rz);
    }
    if (A.cpart) rz += wave_sum_partials<8>(A.cpart + par * A.cnsb, A.cnsb);
    if (f != 0) return;  // uniform over the wavefront
    if (!(pq > 0.0)) {
        if (bid == pb && lane == 0) {
            A.flag[inst] = 2;
            A.scal[3 * inst + 2] = (double)it;
        }
        return;
    }
    const double alpha = rz / pq;
    double drz = 0.0, drr = 0.0;
    if (own) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            A.x[3 * v + i] = xv[i] + alpha * pv[i];
            rv[i] = rv[i] - alpha * qv[i];
            r_out[3 * v + i] = rv[i];
        }
        double zv[3];
        if (cm.y < 0) {
#pragma unroll
            for (int i = 0; i < 3; ++i) zv[i] = o0[3 * i] * rv[0] + o0[3 * i + 1] * rv[1] + o0[3 * i + 2] * rv[2];
        } else {
            // z = M r with the members' updated residuals (the own one as above)
            cl_apply(cm, A.Z, A.nV, v, rv,
                     [&](int u, double* out) {
                         if (u == v) {
                             out[0] = rv[0];
                             out[1] = rv[1];
                             out[2] = rv[2];
                         } else {
#pragma unroll
                             for (int i = 0; i < 3; ++i) out[i] = r_in[3 * u + i] - alpha * A.q[3 * u + i];
                         }
                     },
                     zv);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            A.z[3 * v + i] = zv[i];
            drz += rv[i] * zv[i];
            drr += rv[i] * rv[i];
        }
    }
    drz = wave_sum(drz);
    drr = wave_sum(drr);
    if (lane == 0) {
        A.part_rz[(par ^ 1) * A.nbB + bid] = drz;
        A.part_rr[(par ^ 1) * A.nbB + bid] = drr;
    }
}

// ---------------------------------------------------------------------------
// A whole PCG solve as one kernel.  Each instance's solve is run by a team of
// workgroups that are resident together (or by one); they meet where the two
// kernels above would end, and nothing is launched or read back until the
// solve stops.  Same sums in the same order as those kernels (and
// k_coarse_restrict / k_coarse_solve), so the results are the same bit for
// bit, whatever the team size.
//
// Vectors that other workgroups of the team read (z, p, q, r) go through
// agent-scope relaxed atomic accesses: they reach the memory the eight XCDs
// share without the write-back and invalidation of a whole L2 that a release
// / acquire fence costs, so the matrix, the preconditioner and A_c^-1, read
// with plain loads, stay in each XCD's L2 (or in registers, for the first
// rows of a workgroup) over the iterations.  The workgroups meet on the
// partial sums themselves: a partial is published as two 64-bit words, half
// of its bits and the iteration's tag in each, after every wavefront's vector
// stores were acknowledged, and a reader polls until both tags match.  A
// team of one workgroup (ONE) uses plain accesses and LDS.
// ---------------------------------------------------------------------------
constexpr int TEAM_THREADS = 512;  // 2 wavefronts per SIMD: 256 registers a lane, room for the first rows' blocks
constexpr int TEAM_WAVES = TEAM_THREADS / 64;
constexpr int TEAM_TASKS = 512;    // coarse aggregates at most (and, fewer, wavefront row sums)
constexpr int TEAM_VALUES = 1952;  // values of one meeting at most (r_c of 320 aggregates)

struct TeamArgs {
    const int4* tab;  // per workgroup {instance, rank, team size, 0}; null: one instance, the whole grid
    const int* vbeg;  // instance vertex ranges (B + 1)
    const int* it0;   // per instance: iterations of earlier calls (null: 0)
    // published partials, two words each: p.q (nbA), r.z, r.r and the hand-over mark (2 nbB + B), r_c, r_c . e_c
    unsigned long long *w_pq, *w_r, *w_rc, *w_cp;
    unsigned tag0;    // tags of this launch are tag0 + 1 + iteration; larger than any before
    int* ctl;         // [0] a wait ran out (the launch is void)
    int* done;        // per instance: iterations done by this call when handed over
    int* hand;        // hand-over counts (team_hand): solves past each look, solves stopped before it, solves started
    unsigned* start;  // per instance: workgroups of its team that are resident, TEAM_LEFT when one has left
    long start_limit; // polls of the wait for all of them
    int nstart;       // hand-over: solves at launch (0: never)
    long spin_limit;  // polls of one wait at most
    // coarse level (one instance; K = 0: none)
    int K, ncd, lda, nfree;
    const int *aptr, *avert;
    const double *Ps, *Ainv;
};

template <bool ONE, class T>
__device__ inline T team_ld(const T* p)
{
    if (ONE) return *p;
    return __hip_atomic_load(const_cast<T*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool ONE, class T>
__device__ inline void team_st(T* p, T v)
{
    if (ONE) *p = v;
    else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

typedef unsigned team_u2 __attribute__((ext_vector_type(2)));
typedef unsigned team_u4 __attribute__((ext_vector_type(4)));

__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// ends a phase that stored vectors: every wavefront's stores have reached the
// memory they are read from, then the workgroup's LDS is in step
__device__ inline void team_stores_done()
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

__device__ inline __amdgpu_buffer_rsrc_t team_words(const unsigned long long* w, int n)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned long long*>(w), 0, 16 * n, 0x00027000);
}

// value i of a meeting of n: published (the two words in one store), or (one workgroup) put where team_meet would
template <bool ONE>
__device__ inline void team_put(unsigned long long* w, int n, double* val, int i, double v, unsigned tag)
{
    if (ONE) {
        val[i] = v;
    } else {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        const team_u4 d = {(unsigned)b, tag, (unsigned)(b >> 32), tag};
        __builtin_amdgcn_raw_buffer_store_b128(d, team_words(w, n), 16 * i, 0, 16);
    }
}

// waits for the n values of a meeting and leaves them in val (LDS); false
// when the wait ran out, which voids the launch: every workgroup then leaves
template <bool ONE>
__device__ inline bool team_meet(const TeamArgs& T, const unsigned long long* w, int n, unsigned tag, double* val,
                                 int* bad)
{
    if (!ONE) {
        const __amdgpu_buffer_rsrc_t rs = team_words(w, n);
        constexpr int M = 4;  // values of a thread whose loads are in flight together
        for (int base = 0; base < n; base += M * TEAM_THREADS) {
            team_u4 v[M];
            bool ok = false;
            for (long k = 0; k < T.spin_limit && !ok; ++k) {
                asm volatile("" ::: "memory");  // the loads are made anew in every round
                ok = true;
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const int i = base + (int)threadIdx.x + TEAM_THREADS * m;
                    if (i < n) v[m] = __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * i, 0, 16);
                }
#pragma unroll
                for (int m = 0; m < M; ++m)
                    if (base + (int)threadIdx.x + TEAM_THREADS * m < n) ok = ok && v[m][1] == tag && v[m][3] == tag;
            }
            if (!ok) {
                *bad = 1;
                team_st<false>(T.ctl, 1);
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int i = base + (int)threadIdx.x + TEAM_THREADS * m;
                if (i < n) val[i] = __longlong_as_double((long long)(((unsigned long long)v[m][2] << 32) | v[m][0]));
            }
        }
    }
    __syncthreads();
    return ONE || *bad == 0;
}

// A team starts when all of its workgroups are resident: only then can they
// wait for each other.  Nothing reserves the CUs (a cooperative launch would,
// but only one process can hold that queue), so a workgroup that has waited
// too long for the others leaves, if the team is still incomplete, and then
// all of them do: the solve was not touched and runs in the two-kernel loop.
// (A limit of 0 starts the teams whose workgroups come together, a negative
// one none.)
constexpr unsigned TEAM_LEFT = 0x80000000u;
__device__ inline bool team_start(unsigned* word, unsigned size, long limit)
{
    unsigned w = __hip_atomic_fetch_add(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    for (long k = 0;; ++k) {
        if (w & TEAM_LEFT) return false;
        if (w == size && limit >= 0) return true;
        if (k >= limit && __hip_atomic_compare_exchange_strong(word, &w, w | TEAM_LEFT, __ATOMIC_RELAXED,
                                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return false;  // (on failure w is the word as it stands)
        if (k < limit) w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Whether the solves still running are handed over at look k: as in the
// two-kernel loop, when half of the launch's solves had stopped by then.  That
// loop's solves go in step; here a solve that needs the answer, which is after
// twice as many iterations, may have to wait until every other one is past the
// look or has stopped.  Only solves of which all have started wait: their
// workgroups are resident, the one furthest behind always runs, so the wait
// ends (and is bounded like every other).  The answer does not depend on how
// fast each runs; only where some have not started yet (other work on the GPU)
// is it no, and the solves go on.
__device__ inline bool team_hand(const TeamArgs& T, int k)
{
    if (k >= HAND_LOOKS || team_ld<false>(T.hand + 2 * HAND_LOOKS) != T.nstart) return false;
    for (long n = 0; n < T.spin_limit / HAND_LOOKS; ++n) {
        const int past = team_ld<false>(T.hand + k);
        int stopped = 0;
        for (int j = 0; j <= k; ++j) stopped += team_ld<false>(T.hand + HAND_LOOKS + j);
        if (past + stopped == T.nstart) return 2 * past <= T.nstart;
    }
    return false;
}

// cross-lane moves of a double within a row of 16 lanes (DPP; an LDS
// permute has several times the latency, and these sums are serial)
template <int CTRL, int BANKS>
__device__ inline double dpp_f64(double old, double x)
{
    const long long xi = __double_as_longlong(x), oi = __double_as_longlong(old);
    const int lo = __builtin_amdgcn_update_dpp((int)oi, (int)xi, CTRL, 0xf, BANKS, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(oi >> 32), (int)(xi >> 32), CTRL, 0xf, BANKS, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double dpp_xor1(double x) { return dpp_f64<0xB1, 0xf>(0.0, x); }  // quad_perm 1 0 3 2
__device__ inline double dpp_xor2(double x) { return dpp_f64<0x4E, 0xf>(0.0, x); }  // quad_perm 2 3 0 1
__device__ inline double dpp_xor4(double x) { return dpp_f64<0x124, 0xA>(dpp_f64<0x12C, 0x5>(0.0, x), x); }  // row_ror
__device__ inline double dpp_xor8(double x) { return dpp_f64<0x128, 0xf>(0.0, x); }                          // row_ror:8

// wave_sum with the same partners in the same order (240 clocks instead of 600)
__device__ inline double wave_sum_dpp(double x)
{
    {
        const long long i = __double_as_longlong(x);
        const auto a = __builtin_amdgcn_permlane32_swap((unsigned)i, (unsigned)i, false, false);
        const auto b = __builtin_amdgcn_permlane32_swap((unsigned)(i >> 32), (unsigned)(i >> 32), false, false);
        x = __longlong_as_double(((long long)b[0] << 32) | a[0]) + __longlong_as_double(((long long)b[1] << 32) | a[1]);
    }
    {
        const long long i = __double_as_longlong(x);
        const auto a = __builtin_amdgcn_permlane16_swap((unsigned)i, (unsigned)i, false, false);
        const auto b = __builtin_amdgcn_permlane16_swap((unsigned)(i >> 32), (unsigned)(i >> 32), false, false);
        x = __longlong_as_double(((long long)b[0] << 32) | a[0]) + __longlong_as_double(((long long)b[1] << 32) | a[1]);
    }
    x += dpp_xor8(x);
    x += dpp_xor4(x);
    x += dpp_xor2(x);
    x += dpp_xor1(x);
    return x;
}

// r.z of update block b in the second meeting's values (r.r two further): two
// blocks fill a 64-byte line, a workgroup's own where their number is even.
// Where it is odd most workgroups write halves of two lines (a split that
// gives each its line and the last one the single block was no faster: one
// direction of the 43x11x9 bar 1.33 ms either way, the bent 20x4x4 bar 0.5%
// slower)
__device__ inline int team_rblk(int b) { return 4 * (b >> 1) + (b & 1); }
struct TeamRblk {
    __device__ int operator()(int b) const { return team_rblk(b); }
};

// the order of wave_sum_partials over n values (LDS or global memory)
struct TeamIdent {
    __device__ int operator()(int i) const { return i; }
};
template <class F = TeamIdent>
__device__ inline double team_sum(const double* part, int n, F at = F())
{
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    for (int base = 0; base < n; base += 64 * 8) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i = base + lane + 64 * k;
            v[k] = i < n ? part[at(i)] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) acc += v[k];
    }
    return wave_sum_dpp(acc);
}

// A vector as a buffer resource: its gathers take a 32-bit byte offset (one
// register of address instead of two per load) and two loads per 3-vector.
// Cache policy 16 is sc1, the agent-scope access of team_ld.
struct TeamBuf {
    __amdgpu_buffer_rsrc_t rs;
    __device__ TeamBuf(double* p, long n) : rs(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(unsigned)(8 * n), 0x00027000)) {}
    template <bool ONE>
    __device__ void ld3(unsigned off, unsigned base, double* o) const
    {
        const team_u4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, off, base, ONE ? 0 : 16);
        const team_u2 b = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 16u, base, ONE ? 0 : 16);
        o[0] = __longlong_as_double((long long)(((unsigned long long)a[1] << 32) | a[0]));
        o[1] = __longlong_as_double((long long)(((unsigned long long)a[3] << 32) | a[2]));
        o[2] = __longlong_as_double((long long)(((unsigned long long)b[1] << 32) | b[0]));
    }
    template <bool ONE>
    __device__ double ld1(unsigned off, unsigned base) const
    {
        const team_u2 b = __builtin_amdgcn_raw_buffer_load_b64(rs, off, base, ONE ? 0 : 16);
        return __longlong_as_double((long long)(((unsigned long long)b[1] << 32) | b[0]));
    }
};

// one BSR block of a row: slot j of its elastic blocks followed by its
// contact blocks, and its column.  A slot past the row's end is a zero block
// on the row itself (no branch; it adds 0).
struct TeamSlot {
    int col;
    double b[9];
    __device__ void load(const PcgArgs& A, int v, int j, int e0, int ne, int c0, int nc)
    {
        col = v;
#pragma unroll
        for (int e = 0; e < 9; ++e) b[e] = 0.0;
        if (j >= ne + nc) return;
        const bool el = j < ne;
        const double* __restrict__ val = el ? A.eval : A.cval;
        const long ld = el ? A.eld : A.cld;
        const int k = el ? e0 + j : c0 + (j - ne);
        col = el ? A.ecol[k] : A.ccol[k];
#pragma unroll
        for (int e = 0; e < 9; ++e) b[e] = val[e * ld + k];
    }
};

// The columns of a workgroup's rows, each once: a set over the instance's
// vertices (one bit each, with the number of members before each word) and
// its members in order.  Every iteration reads z and p_old of the first
// TEAM_COLS members into LDS once, instead of once per block that uses them:
// a lane's gather of a 24-byte record occupies the CU's address unit for a
// whole cache line, and 128 rows of about 14 blocks have some 500 columns
// (row phase of the 64x16x16 bar: 4.2 us with one gather per block).
constexpr int TEAM_COLS = 1024;
constexpr int TEAM_SET = TEAM_MAX * TEAM_ROWS / 32;  // words of a set
struct TeamCols {
    unsigned* bits;
    int* before;
    int* list;
    double *z, *p;  // 3 per member
    __device__ int find(int c) const
    {
        const unsigned w = bits[c >> 5];
        return before[c >> 5] + __popc(w & ((1u << (c & 31)) - 1u));
    }
};

struct TeamVec {
    double z[3], p[3];
    // z and p_old (byte po of the p buffer) at column col, member k of the set
    template <bool ONE>
    __device__ void load(const TeamBuf& bz, const TeamBuf& bp, unsigned po, const TeamCols& C, int k, int col)
    {
        if (k < TEAM_COLS) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                z[d] = C.z[3 * k + d];
                p[d] = C.p[3 * k + d];
            }
        } else {
            bz.ld3<ONE>(24u * (unsigned)col, 0, z);
            bp.ld3<ONE>(24u * (unsigned)col, po, p);
        }
    }
    // y += B z, w += B p (row_spmv's sums)
    __device__ void add(const TeamSlot& S, double* y, double* w) const
    {
#pragma unroll
        for (int i = 0; i < 3; ++i) y[i] += S.b[3 * i] * z[0] + S.b[3 * i + 1] * z[1] + S.b[3 * i + 2] * z[2];
#pragma unroll
        for (int i = 0; i < 3; ++i) w[i] += S.b[3 * i] * p[0] + S.b[3 * i + 1] * p[1] + S.b[3 * i + 2] * p[2];
    }
};

// what a lane of the update keeps of its row: lane b of a row's four holds
// the row's preconditioner block for cluster member b and that member's
// residual (every holder of a residual updates it alike); the lane of the row
// itself also holds x
struct TeamRow {
    int v, u;  // row, member (-1: none)
    bool own, single;
    double Z[9], r[3], x[3];
    template <bool ONE>
    __device__ void load(const PcgArgs& A, int row, int vend, int b, const double* r_in)
    {
        v = row;
        u = -1;
        own = single = false;
#pragma unroll
        for (int e = 0; e < 9; ++e) Z[e] = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) r[d] = x[d] = 0.0;
        if (v >= vend) return;
        const int4 cm = A.cm4[v];
        single = cm.y < 0;
        u = b == 0 ? cm.x : b == 1 ? cm.y : b == 2 ? cm.z : cm.w;
        if (single && b == 0) u = v;
        if (u < 0) return;
        own = u == v;
        const double* o = A.Z + 9 * ((size_t)b * A.nV + v);
#pragma unroll
        for (int e = 0; e < 9; ++e) Z[e] = o[e];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            r[d] = team_ld<ONE>(r_in + 3 * (size_t)u + d);
            if (own) x[d] = A.x[3 * (size_t)v + d];
        }
    }
};

// a row's block count and its first two slots of this lane (rows past the end: zero blocks on row v0)
struct TeamTask {
    int n, ka, kb, ko;  // blocks of the row; members of the column set of the two slots and of the row
    TeamSlot a, b;
    __device__ void load(const PcgArgs& A, int v, int vend, int v0, int gl)
    {
        int e0 = 0, ne = 0, c0 = 0, nc = 0;
        if (v < vend) row_extents(A, v, e0, ne, c0, nc);
        else v = v0;
        n = ne + nc;
        a.load(A, v, gl, e0, ne, c0, nc);
        b.load(A, v, gl + 8, e0, ne, c0, nc);
    }
};

// p and q = A p of row v (8 lanes, row_spmv's order); the wavefront's sum of p.q
template <bool ONE>
__device__ inline double team_row(const PcgArgs& A, const TeamBuf& bz, const TeamBuf& bp, unsigned po, const TeamCols& C,
                                  const TeamTask& K, int v, int vend, int v0, int gl, double beta, double* pn)
{
    double y[3] = {0.0, 0.0, 0.0}, w[3] = {0.0, 0.0, 0.0};
    double zo, poo;  // this lane's component of the row's own z and p_old
    {
        TeamVec Va, Vb;
        Va.load<ONE>(bz, bp, po, C, K.ka, K.a.col);
        Vb.load<ONE>(bz, bp, po, C, K.kb, K.b.col);
        const int g = min(gl, 2);
        if (K.ko < TEAM_COLS) {
            zo = C.z[3 * K.ko + g];
            poo = C.p[3 * K.ko + g];
        } else {
            const unsigned i = 24u * (unsigned)(v < vend ? v : v0) + 8u * (unsigned)g;
            zo = bz.ld1<ONE>(i, 0);
            poo = bp.ld1<ONE>(i, po);
        }
        Va.add(K.a, y, w);
        Vb.add(K.b, y, w);
    }
    if (K.n > 16) {  // longer rows: the rest of their blocks from memory
        int e0, ne, c0, nc;
        row_extents(A, v, e0, ne, c0, nc);
        for (int j = gl + 16; j < K.n; j += 8) {
            TeamSlot S;
            TeamVec u;
            S.load(A, v, j, e0, ne, c0, nc);
            u.load<ONE>(bz, bp, po, C, C.find(S.col - v0), S.col);
            u.add(S, y, w);
        }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) y[i] += beta * w[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) y[i] += dpp_xor4(y[i]);
#pragma unroll
    for (int i = 0; i < 3; ++i) y[i] += dpp_xor2(y[i]);
#pragma unroll
    for (int i = 0; i < 3; ++i) y[i] += dpp_xor1(y[i]);
    double yl = y[2];
    yl = gl == 1 ? y[1] : yl;
    yl = gl == 0 ? y[0] : yl;
    double d = 0.0;
    if (gl < 3 && v < vend) {
        const size_t i = 3 * (size_t)v + gl;
        const double pv = zo + beta * poo;
        team_st<ONE>(pn + i, pv);
        team_st<ONE>(A.q + i, yl);
        d = pv * yl;
    }
    return wave_sum_dpp(d);
}

// COARSE: with the coarse level (T.K > 0); HAND: solves may be handed over
// (T.nstart > 0, never with the coarse level).  Variants of their own, since
// the registers are full: the hand-over's few values cost the twisted 64x16x16
// bar 1.6% of its step in spills.
template <bool ONE, bool COARSE, bool HAND>
__global__ void __launch_bounds__(TEAM_THREADS) k_pcg_team(PcgArgs A, TeamArgs T)
{
    __shared__ double wt[TEAM_TASKS];
    __shared__ double val[TEAM_VALUES];
    __shared__ double rowz[TEAM_ROWS], rowr[TEAM_ROWS];
    __shared__ unsigned cbits[TEAM_SET];
    __shared__ int cbefore[TEAM_SET], clist[TEAM_COLS];
    __shared__ double cz[3 * TEAM_COLS], cp[3 * TEAM_COLS];
    const TeamCols C{cbits, cbefore, clist, cz, cp};
    __shared__ double sh[8];
    __shared__ double shc[TEAM_WAVES][6];
    __shared__ int bad, cwave[TEAM_WAVES];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int inst = 0, rank = blockIdx.x, size = gridDim.x;
    if (T.tab) {
        const int4 t = T.tab[blockIdx.x];
        inst = uni(t.x);
        rank = uni(t.y);
        size = uni(t.z);
    }
    if (!ONE && size > 1) {
        if (tid == 0) bad = team_start(T.start + inst, (unsigned)size, T.start_limit) ? 0 : 1;
        __syncthreads();
        if (bad) return;
    }
    const int v0 = uni(T.vbeg[inst]), v1 = uni(T.vbeg[inst + 1]);
    const int pb = uni(A.bpbeg[inst]), nb = uni(A.bpbeg[inst + 1]) - pb;
    const int ab = uni(A.apbeg[inst]), na = uni(A.apbeg[inst + 1]) - ab;
    // this workgroup's 64-row update blocks and the 32-row SpMV blocks of the same rows
    const int b0 = (int)((long)nb * rank / size), b1 = (int)((long)nb * (rank + 1) / size);
    const int u0 = 2 * b0, nu = min(2 * b1, na) - u0;
    const int rb = v0 + 64 * b0, re = min(v0 + 64 * b1, v1);
    const int it_first = T.it0 ? uni(T.it0[inst]) : 0;
    const TeamBuf bz(A.z, 3L * A.nV), bp(A.pbuf, 6L * A.nV), bq(A.q, 3L * A.nV), br(A.r, 6L * A.nV);
    unsigned long long* w_pq = T.w_pq + 2 * (size_t)ab;
    const int nr = 4 * ((nb + 1) / 2) + 1;  // values of the second meeting; the last: the hand-over mark
    unsigned long long* w_r = T.w_r + 2 * (2 * (size_t)pb + 8 * inst);
    double* sci = A.scal + 3 * inst;
    double rz = 0.0, rr = 0.0, rzo = 1.0, bb = 0.0;
    int hand = 0;
    // hand-over, by one thread of the solve: its next look (and which), the next look whose answer it needs
    __shared__ int look[2], ans[2];
    const bool counts = HAND && rank == 0 && tid == 0;
    if (counts) {
        look[0] = ans[0] = HAND_FIRST;
        look[1] = ans[1] = 0;
        atomicAdd(T.hand + 2 * HAND_LOOKS, 1);
    }
    if (tid == 0) bad = 0;
    // ---- the workgroup's blocks and update state stay in registers
    const int gl = lane & 7;
    const int row0 = rb + 8 * wave + (lane >> 3);  // SpMV rows: row0 and row0 + 64
    TeamTask K0, K1;
    K0.load(A, row0, re, v0, gl);
    K1.load(A, row0 + 64, re, v0, gl);
    int ncol = 0;
    {
        const int nw = (v1 - v0 + 31) >> 5;
        for (int i = tid; i < nw; i += TEAM_THREADS) cbits[i] = 0u;
        __syncthreads();
        auto mark = [&](int col) { atomicOr(&cbits[(col - v0) >> 5], 1u << ((col - v0) & 31)); };
        for (int k = 0; k < 2; ++k) {
            const int v = row0 + 64 * k;
            if (v >= re) continue;
            int e0, ne, c0, nc;
            row_extents(A, v, e0, ne, c0, nc);
            for (int j = gl; j < ne + nc; j += 8) mark(j < ne ? A.ecol[e0 + j] : A.ccol[c0 + j - ne]);
        }
        if (tid == 0) mark(v0);  // where the lanes past the rows' end point
        __syncthreads();
        // members before each word: a run of words per thread, then the runs' sums
        const int per = (nw + TEAM_THREADS - 1) / TEAM_THREADS;
        const int w0 = min(tid * per, nw), w1 = min(w0 + per, nw);
        int cnt = 0;
        for (int i = w0; i < w1; ++i) cnt += __popc(cbits[i]);
        int inc = cnt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(inc, o, 64);
            if (lane >= o) inc += t;
        }
        if (lane == 63) cwave[wave] = inc;
        __syncthreads();
        int at = inc - cnt;
        for (int w = 0; w < TEAM_WAVES; ++w) {
            if (w < wave) at += cwave[w];
            ncol += cwave[w];
        }
        for (int i = w0; i < w1; ++i) {
            cbefore[i] = at;
            for (unsigned b = cbits[i]; b; b &= b - 1u) {
                if (at < TEAM_COLS) clist[at] = v0 + 32 * i + __ffs((int)b) - 1;
                ++at;
            }
        }
        __syncthreads();
        ncol = min(uni(ncol), TEAM_COLS);
        K0.ka = C.find(K0.a.col - v0);
        K0.kb = C.find(K0.b.col - v0);
        K1.ka = C.find(K1.a.col - v0);
        K1.kb = C.find(K1.b.col - v0);
        K0.ko = C.find((row0 < re ? row0 : v0) - v0);
        K1.ko = C.find((row0 + 64 < re ? row0 + 64 : v0) - v0);
    }
    const int ur = 16 * wave + (lane >> 2), ub = lane & 3;  // update: row, cluster member
    TeamRow R0;
    R0.load<true>(A, rb + ur, re, ub, A.r + (size_t)(it_first & 1) * 3 * A.nV);
    // ---- the sums that the launch starts from
    {
        const int par = it_first & 1;
        double s = 0.0;
        if (wave == 0) s = team_sum(A.part_rz + par * A.nbB + pb, nb);
        else if (wave == 1) s = team_sum(A.part_rr + par * A.nbB + pb, nb);
        else if (wave == 2 && COARSE) s = team_sum(A.cpart + par * T.K, T.K);
        else if (wave == 3) s = team_sum(it_first > 0 ? A.part_rz + (par ^ 1) * A.nbB + pb : A.part_rr + A.nbB + pb, nb);
        if (wave < 4 && lane == 0) sh[wave] = s;
        __syncthreads();
        rz = sh[0];
        rr = sh[1];
        if (COARSE) rz += sh[2];
        if (it_first > 0) {
            rzo = sh[3];
            bb = sci[0];
        } else {
            bb = sh[3];
        }
    }
    int state = 0;  // 1 converged, 4 iteration limit, 2 breakdown, -1 handed over
    int it = it_first;
    for (;; ++it) {
        const unsigned tag = T.tag0 + 1u + (unsigned)(it - it_first);
        const int par = it & 1;
        // the same decisions in every workgroup of the team
        if (HAND && hand) {
            state = -1;
            break;
        }
        if (counts && it - it_first == look[0]) {
            if (look[1] < HAND_LOOKS) atomicAdd(T.hand + look[1], 1);
            look[0] = hand_next(look[0]);
            ++look[1];
        }
        if (!(bb > 0.0) || (it > 0 && rr <= A.rtol2 * bb)) {
            state = 1;
            break;
        }
        if (it >= A.maxit) {
            state = 4;
            break;
        }
        const double beta = it > 0 ? rz / rzo : 0.0;
        rzo = rz;
        // ---- p = z + beta p_old, q = A p and the partials of p.q
        const unsigned po = (unsigned)(par ^ 1) * 24u * (unsigned)A.nV;  // p_old is zero at iteration 0
        const unsigned pc = (unsigned)par * 24u * (unsigned)A.nV;
        double* pn = A.pbuf + (size_t)par * 3 * A.nV;
        for (int i = tid; i < ncol; i += TEAM_THREADS) {
            const unsigned off = 24u * (unsigned)clist[i];
            bz.ld3<ONE>(off, 0, cz + 3 * i);
            bp.ld3<ONE>(off, po, cp + 3 * i);
        }
        __syncthreads();
        {
            const double da = team_row<ONE>(A, bz, bp, po, C, K0, row0, re, v0, gl, beta, pn);
            const double db = team_row<ONE>(A, bz, bp, po, C, K1, row0 + 64, re, v0, gl, beta, pn);
            if (lane == 0) {
                wt[wave] = da;
                wt[8 + wave] = db;
            }
        }
        team_stores_done();
        if (tid < nu) {
            double a = 0.0;
#pragma unroll
            for (int k = 0; k < 4; ++k) a += wt[4 * tid + k];
            team_put<ONE>(w_pq, na, val, u0 + tid, a, tag);
        }
        if (!team_meet<ONE>(T, w_pq, na, tag, val, &bad)) return;
        // ---- alpha, x, r, z = M r and the partials of r.z, r.r
        double* r_out = A.r + (size_t)(par ^ 1) * 3 * A.nV;
        double q[3] = {0.0, 0.0, 0.0}, pv[3] = {0.0, 0.0, 0.0};
        if (R0.u >= 0) {
            bq.ld3<ONE>(24u * (unsigned)R0.u, 0, q);
            if (R0.own) bp.ld3<ONE>(24u * (unsigned)R0.u, pc, pv);
        }
        if (wave == 0) {
            const double s = team_sum(val, na);
            if (lane == 0) sh[4] = s;
        }
        __syncthreads();
        const double pq = sh[4];
        if (!(pq > 0.0)) {
            state = 2;
            break;
        }
        const double alpha = rz / pq;
        {
            double t[3], zv[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) R0.r[d] = R0.r[d] - alpha * q[d];
#pragma unroll
            for (int d = 0; d < 3; ++d)
                t[d] = R0.Z[3 * d] * R0.r[0] + R0.Z[3 * d + 1] * R0.r[1] + R0.Z[3 * d + 2] * R0.r[2];
            // the members' terms in order (every lane of the row gets the sum)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double t0 = dpp_f64<0x00, 0xf>(0.0, t[d]), t1 = dpp_f64<0x55, 0xf>(0.0, t[d]),
                             t2 = dpp_f64<0xAA, 0xf>(0.0, t[d]), t3 = dpp_f64<0xFF, 0xf>(0.0, t[d]);
                zv[d] = R0.single ? t0 : ((t0 + t1) + t2) + t3;
            }
            if (R0.own) {
                const size_t i0 = 3 * (size_t)R0.v;
                double drz = 0.0, drr = 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    R0.x[d] = R0.x[d] + alpha * pv[d];
                    team_st<ONE>(r_out + i0 + d, R0.r[d]);
                    team_st<ONE>(A.z + i0 + d, zv[d]);
                    drz += R0.r[d] * zv[d];
                    drr += R0.r[d] * R0.r[d];
                }
                rowz[ur] = drz;
                rowr[ur] = drr;
            } else if (ub == 0 && R0.v >= re) {
                rowz[ur] = rowr[ur] = 0.0;
            }
        }
        team_stores_done();
        // the workgroup's (at most) two 64-row blocks; lanes 0..3 publish their r.z and r.r together
        if (wave == 0) {
            const double z0 = wave_sum_dpp(rowz[lane]), z1 = wave_sum_dpp(rowz[64 + lane]);
            const double q0 = wave_sum_dpp(rowr[lane]), q1 = wave_sum_dpp(rowr[64 + lane]);
            const int blk = b0 + (lane & 1);
            if (lane < 4 && blk < b1) {
                const double s = lane < 2 ? (lane ? z1 : z0) : (lane & 1 ? q1 : q0);
                // for a call that continues this solve
                (lane < 2 ? A.part_rz : A.part_rr)[(par ^ 1) * A.nbB + pb + blk] = s;
                team_put<ONE>(w_r, nr, val, team_rblk(blk) + (lane & 2), s, tag);
            }
        }
        // an odd number of blocks: the last line's other half is published too, so that all of it is waited for
        if (wave == 1 && lane < 2 && (nb & 1) && rank == size - 1)
            team_put<ONE>(w_r, nr, val, team_rblk(nb) + 2 * lane, 0.0, tag);
        if (counts) {
            double mark = 0.0;
            if (it + 1 - it_first == 2 * ans[0]) {
                if (team_hand(T, ans[1])) mark = 1.0;
                ans[0] = hand_next(ans[0]);
                ++ans[1];
            }
            team_put<ONE>(w_r, nr, val, nr - 1, mark, tag);
        }
        if (!team_meet<ONE>(T, w_r, HAND ? nr : nr - 1, tag, val, &bad)) return;
        if (wave == 0) {
            const double s = team_sum(val, nb, TeamRblk());
            if (lane == 0) sh[0] = s;
        } else if (wave == 1) {
            const double s = team_sum(val + 2, nb, TeamRblk());
            if (lane == 0) sh[1] = s;
        } else if (HAND && wave == 2 && lane == 0) {
            sh[5] = val[nr - 1];
        }
        if (COARSE) {
            __syncthreads();  // val is read above and written by the next meeting
            // ---- coarse level: r_c = P^T r, then e_c = A_c^-1 r_c and z += P e_c; 256 threads per aggregate
            const int q4 = tid >> 8, t4 = tid & 255;
            for (int a0 = rank; a0 < T.K; a0 += 2 * size) {
                const int a = a0 + q4 * size;
                double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                if (a < T.K) {
                    const int j1 = T.aptr[a + 1];
                    for (int j = T.aptr[a] + t4; j < j1; j += 256) {
                        double x[3], Pv[18];
                        br.ld3<ONE>(24u * (unsigned)T.avert[j], (unsigned)(par ^ 1) * 24u * (unsigned)A.nV, x);
#pragma unroll
                        for (int m = 0; m < 18; ++m) Pv[m] = T.Ps[(size_t)m * T.nfree + j];
#pragma unroll
                        for (int m = 0; m < 6; ++m) acc[m] += Pv[m] * x[0] + Pv[6 + m] * x[1] + Pv[12 + m] * x[2];
                    }
                }
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    const double s = wave_sum_dpp(acc[m]);
                    if (lane == 0) shc[wave][m] = s;
                }
                __syncthreads();
                if (a < T.K && t4 < 6) {
                    double s = 0.0;
#pragma unroll
                    for (int k = 0; k < 4; ++k) s += shc[4 * q4 + k][t4];
                    team_put<ONE>(T.w_rc, T.ncd, val, 6 * a + t4, s, tag);
                }
                __syncthreads();
            }
            if (!team_meet<ONE>(T, T.w_rc, T.ncd, tag, val, &bad)) return;
            for (int a0 = rank; a0 < T.K; a0 += 2 * size) {
                const int a = a0 + q4 * size;
                double e[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                if (a < T.K) {
                    const double* Ar = T.Ainv + (size_t)(6 * a) * T.lda;
#pragma unroll 4
                    for (int j = t4; j < T.ncd; j += 256) {
                        const double rj = val[j];
#pragma unroll
                        for (int m = 0; m < 6; ++m) e[m] += Ar[(size_t)m * T.lda + j] * rj;
                    }
                }
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    const double s = wave_sum_dpp(e[m]);
                    if (lane == 0) shc[wave][m] = s;
                }
                __syncthreads();
                if (a < T.K) {
#pragma unroll
                    for (int m = 0; m < 6; ++m) {
                        double s = 0.0;
#pragma unroll
                        for (int k = 0; k < 4; ++k) s += shc[4 * q4 + k][m];
                        e[m] = s;
                    }
                    if (t4 == 0) {
                        double d = 0.0;
#pragma unroll
                        for (int m = 0; m < 6; ++m) d += val[6 * a + m] * e[m];
                        wt[a] = d;
                    }
                    const int j1 = T.aptr[a + 1];
                    for (int j = T.aptr[a] + t4; j < j1; j += 256) {
                        const int v = T.avert[j];
                        double x[3], Pv[18];
                        bz.ld3<ONE>(24u * (unsigned)v, 0, x);
#pragma unroll
                        for (int m = 0; m < 18; ++m) Pv[m] = T.Ps[(size_t)m * T.nfree + j];
#pragma unroll
                        for (int d = 0; d < 3; ++d) {
                            double s = 0.0;
#pragma unroll
                            for (int m = 0; m < 6; ++m) s += Pv[6 * d + m] * e[m];
                            team_st<ONE>(A.z + 3 * (size_t)v + d, x[d] + s);
                        }
                    }
                }
                __syncthreads();
            }
            team_stores_done();
            for (int a = rank + tid * size; a < T.K; a += TEAM_THREADS * size) team_put<ONE>(T.w_cp, T.K, val, a, wt[a], tag);
            if (!team_meet<ONE>(T, T.w_cp, T.K, tag, val, &bad)) return;
            if (wave == 0) {
                const double s = team_sum(val, T.K);
                if (lane == 0) sh[2] = s;
            }
        }
        __syncthreads();
        rz = sh[0];
        rr = sh[1];
        if (HAND) hand = sh[5] != 0.0;
        if (COARSE) rz += sh[2];
    }
    // ---- the solve stopped or is handed over
    if (R0.own && it > it_first)
#pragma unroll
        for (int d = 0; d < 3; ++d) A.x[3 * (size_t)R0.v + d] = R0.x[d];
    if (rank != 0 || tid != 0) return;
    if (state != 2) sci[0] = bb;
    if (state == -1) {  // the state is on the device: a later call continues at this iteration
        T.done[inst] = it - it_first;
        return;
    }
    A.flag[inst] = state;
    if (state != 2) sci[1] = rr;
    sci[2] = (double)it;
    if (counts && look[1] < HAND_LOOKS) atomicAdd(T.hand + HAND_LOOKS + look[1], 1);  // stopped before its next look
}

// generic deterministic sum of partials -> out[0]
__global__ void __launch_bounds__(RB) k_sum_partials(int npart, const double* __restrict__ part,
                                                     double* __restrict__ out)
{
    __shared__ double sh[RB];
    const double s = sum_partials_block(part, npart, sh);
    if (threadIdx.x == 0) out[0] = s;
}

// x = a + s * b
__global__ void k_axpy3(long n, const double* __restrict__ a, double s, const double* __restrict__ b,
                        double* __restrict__ x)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    x[i] = a[i] + s * b[i];
}

// v = (x - xn) / h  (IMPLICIT_EULER.h:882-888)
__global__ void k_velocity(long n, const double* __restrict__ x, const double* __restrict__ xn, double h,
                           double* __restrict__ v)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    v[i] = (x[i] - xn[i]) / h;
}

// partial sums of a.b
__global__ void __launch_bounds__(RB) k_dot_parts(long n, const double* __restrict__ a,
                                                  const double* __restrict__ b, double* __restrict__ part)
{
    __shared__ double sh[RB];
    long i = (long)blockIdx.x * RB + threadIdx.x;
    double d = (i < n) ? a[i] * b[i] : 0.0;
    double s = block_sum<RB>(d, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {
unsigned read_u(PinBuf& pin, hipStream_t s, const unsigned* p)
{
    unsigned* v = pin.as<unsigned>(1);
    IDP_HIP(hipMemcpyAsync(v, p, sizeof(unsigned), hipMemcpyDeviceToHost, s));
    IDP_HIP(hipStreamSynchronize(s));
    return *v;
}
int bits_for(unsigned long long maxv)
{
    int b = 1;
    while (b < 64 && (maxv >> b)) ++b;
    return b;
}
}  // namespace

void contact_structure(LinWork& L, hipStream_t s, int nV, long ncs0, const int* cs, long nf, const int* fcs)
{
    L.ncb = 0;
    L.nrec = 0;
    const long ncs = ncs0 + nf;
    if (ncs == 0) return;
    if (ncs >= (1L << 24)) throw std::length_error("contact structure: more than 2^24 stencils");
    int* vid = L.vid.ensure(4 * (size_t)ncs, s);
    int* nv = L.nv.ensure(ncs, s);
    if (ncs0) launch_constraint_vids(s, ncs0, cs, vid, nv);
    if (nf) launch_constraint_vids(s, nf, fcs, vid + 4 * ncs0, nv + ncs0);
    unsigned* cnt = L.u0.ensure(ncs + 1, s);
    unsigned* off = L.u1.ensure(ncs + 1, s);
    IDP_LAUNCH(k_contact_nv2, grid_for(ncs, 256), 256, 0, s, ncs, nv, cnt);
    IDP_HIP(hipMemsetAsync(cnt + ncs, 0, sizeof(unsigned), s));
    excl_scan<unsigned>(s, L.tmp, cnt, off, (int)ncs + 1);
    unsigned nrec = read_u(*L.pin, s, off + ncs);
    unsigned long long V = (unsigned long long)nV;
    unsigned long long* k0 = L.key0.ensure(nrec, s);
    unsigned* v0 = L.rv0.ensure(nrec, s);
    IDP_LAUNCH(k_contact_keys, grid_for(ncs, 256), 256, 0, s, ncs, vid, nv, off, V, k0, v0);
    unsigned long long* k1 = L.key1.ensure(nrec, s);
    unsigned* v1 = L.rv1.ensure(nrec, s);
    sort_pairs(s, L.tmp, k0, k1, v0, v1, nrec, bits_for(V * V));
    unsigned* head = L.u0.ensure(nrec + 1, s);
    unsigned* hs = L.u1.ensure(nrec + 1, s);
    IDP_LAUNCH(k_run_heads, grid_for(nrec + 1, 256), 256, 0, s, nrec, k1, head);
    excl_scan<unsigned>(s, L.tmp, head, hs, (int)nrec + 1);
    unsigned nb = read_u(*L.pin, s, hs + nrec);
    unsigned* seg = L.seg.ensure(nb + 1, s);
    int* crow = L.crow.ensure(nb + 1, s);
    int* ccol = L.ccol.ensure(nb + 1, s);
    int* cdiag = L.cdiag.ensure(nV, s);
    IDP_HIP(hipMemsetAsync(cdiag, 0xff, sizeof(int) * nV, s));
    IDP_LAUNCH(k_contact_pattern, grid_for(nrec, 256), 256, 0, s, nrec, k1, hs, V, nb, seg, crow, ccol, cdiag);
    int* crp = L.crp.ensure(nV + 1, s);
    IDP_LAUNCH(k_rowptr_from_rows, grid_for(nV + 1, 256), 256, 0, s, nb, crow, nV, crp);
    L.ncb = nb;
    L.nrec = nrec;
    L.ncs = ncs;
}

void contact_gradient_gather(LinWork& L, hipStream_t s, const MeshDev& m, const double* X, const double* Xt,
                             const double* gl, const double* gb, double* g, double* rhs, const unsigned char* act)
{
    bool haveC = L.ncb > 0 && gb;
    IDP_LAUNCH(k_gradient_gather, grid_for(m.nV, 256), 256, 0, s, m.nV, m.e_diag.p, m.e_src_ptr.p, m.e_src.p, gl, X,
               Xt, m.mass.p, haveC ? L.cdiag.p : (const int*)nullptr, L.seg.p, L.rv1.p, gb, m.proj_mask(),
               m.inst.vinst.p, act, g, rhs);
}

void assemble(LinWork& L, hipStream_t s, const MeshDev& m, const double* Hl, const double* Hb, bool any_dbc,
              const unsigned char* act)
{
    // algorithmic bytes: 80 per contribution (9 doubles + key), 76 per block, rowptr
    const double ncontrib = 16.0 * m.nT + 9.0 * m.nE + (double)L.nrec + m.nV;
    const int tok = L.prof ? L.prof->begin(IDP_K_ASSEMBLY) : -1;
    double* ev = L.evals.ensure(9 * (size_t)m.nnzb_e, s);
    IDP_LAUNCH(k_elastic_values, grid_for(m.nnzb_e, 256), 256, 0, s, m.nnzb_e, L.erow.p, m.e_col.p, m.e_src_ptr.p,
               m.e_src.p, Hl, m.mass.p, m.inst.vinst.p, act, ev);
    if (L.ncb) {
        double* cv = L.cvals.ensure(9 * (size_t)L.ncb, s);
        IDP_LAUNCH(k_contact_values, grid_for(L.ncb, 256), 256, 0, s, (unsigned)L.ncb, L.seg.p, L.rv1.p, Hb, L.crow.p,
                   m.inst.vinst.p, act, cv);
    }
    if (any_dbc) {
        IDP_LAUNCH(k_project_dbc, grid_for(m.nnzb_e, 256), 256, 0, s, m.nnzb_e, L.erow.p, m.e_col.p, m.proj_mask(), 1,
                   ev);
        if (L.ncb)
            IDP_LAUNCH(k_project_dbc, grid_for(L.ncb, 256), 256, 0, s, (long)L.ncb, L.crow.p, L.ccol.p, m.proj_mask(), 0,
                       L.cvals.p);
    }
    if (L.prof)
        L.prof->end(IDP_K_ASSEMBLY, tok, 80.0 * ncontrib + 76.0 * ((double)m.nnzb_e + L.ncb) + 4.0 * (m.nV + 1));
}

void build_inst_layout(MeshDev& m, const std::vector<long>& vbeg, const std::vector<long>& tbeg,
                       const std::vector<long>& nbeg, const std::vector<long>& ebeg, const std::vector<long>& fbeg,
                       hipStream_t s)
{
    InstDev& I = m.inst;
    I.B = (int)vbeg.size() - 1;
    I.vbeg = vbeg;
    I.tbeg = tbeg;
    I.nbeg = nbeg;
    I.ebeg = ebeg;
    I.fbeg = fbeg;
    std::vector<int> vi(std::max<long>(vbeg.back(), 1), 0);
    for (int i = 0; i < I.B; ++i)
        for (long v = vbeg[i]; v < vbeg[i + 1]; ++v) vi[v] = i;
    I.vinst.upload(vi.data(), vi.size(), s);
    auto up = [&](DBuf<int>& d, const std::vector<long>& h) {
        std::vector<int> t(h.begin(), h.end());
        d.upload(t.data(), t.size(), s);
    };
    up(I.d_vbeg, vbeg);
    up(I.d_nbeg, nbeg);
    up(I.d_ebeg, ebeg);
    up(I.d_fbeg, fbeg);
    I.echunk.build(ebeg, 256, s);
    I.vblk.build(vbeg, RB, s);
    I.nblk.build(nbeg, RB, s);
    I.tblk.build(tbeg, RB, s);
    for (int gi = 0; gi < 4; ++gi) I.pcg_rows[gi].build(vbeg, spmv_rows(4 << gi), s);
    I.pcg_upd.build(vbeg, 64, s);
    std::vector<long> v3(vbeg.size());
    for (size_t i = 0; i < vbeg.size(); ++i) v3[i] = 3 * vbeg[i];
    I.dblk.build(v3, RB, s);
    IDP_HIP(hipStreamSynchronize(s));
}

void init_erow(LinWork& L, hipStream_t s, const MeshDev& m, const std::vector<int>& rowof)
{
    L.erow.upload(rowof.data(), rowof.size(), s);
}

__global__ void k_zero_words(long n, unsigned long long* __restrict__ w)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) w[i] = 0ull;
}

// also clears the team kernel's words (nteam of them)
__global__ void k_pcg_start(int B, const unsigned char* __restrict__ solve, int* __restrict__ flag,
                            int* __restrict__ err, int nteam, int* __restrict__ team)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nteam) team[i] = 0;
    if (i >= B) return;
    flag[i] = (solve && !solve[i]) ? 3 : 0;  // new and continued solves iterate
    err[i] = 0;
}

// workgroups of k_pcg_team that the context's device holds at once
int team_resident()
{
    int dev = 0, cus = 0, per = INT_MAX;
    IDP_HIP(hipGetDevice(&dev));
    IDP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    for (const void* fn : {(const void*)k_pcg_team<false, false, false>, (const void*)k_pcg_team<false, true, false>,
                           (const void*)k_pcg_team<false, false, true>}) {
        int n = 0;
        IDP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, TEAM_THREADS, 0));
        per = std::min(per, n);
    }
    return per * cus;
}

// Runs the solves of the instances in `run` with k_pcg_team; false where the
// two-kernel loop is used instead:
//  - more rows than TEAM_MAX workgroups hold (32,768).  With the rest of the
//    rows read from memory an iteration of 24 cubes (41,580 rows) took 18 us,
//    against 15 us in the two kernels;
//  - a coarse level of more than two aggregates per workgroup and 256-thread
//    half (a sheet of 625 free vertices cut into 320 aggregates, 32 for each of
//    its 10 workgroups, took 1.2 ms more per solve than the four kernels);
//  - launches whose teams the device cannot hold together, contexts of more
//    vertices than 32-bit offsets reach, and, for a while, contexts whose teams
//    found the device taken (team_rule.hpp).
// Below, per iteration and with launch gaps: 81 rows 24 -> 5 us, 18,785 rows
// with 100-130 aggregates 40 -> 30-39 us.
bool pcg_team(LinWork& L, hipStream_t s, const InstDev& I, const PcgArgs& A, const std::vector<char>& run, int* team,
              bool coarse, bool handover)
{
    const int B = I.B;
    std::vector<int4>& tab = L.h_team_tab;  // kept: its upload may be under way when this returns
    tab.clear();
    bool one = true;
    int nrun = 0;
    for (int i = 0; i < B; ++i)
        if (run[i]) {
            ++nrun;
            const int nb = I.pcg_upd.h_pbeg[i + 1] - I.pcg_upd.h_pbeg[i];
            const int t = (nb + 1) / 2;  // TEAM_ROWS rows per workgroup
            if (tab.size() + t > TEAM_MAX) return false;
            for (int k = 0; k < t; ++k) tab.push_back(make_int4(i, k, t, 0));
            one = one && t == 1;
        }
    if (nrun == 0 || !team_addresses(A.nV)) return false;
    if (L.team_resident < 0) L.team_resident = team_resident();
    if (!team_fits((int)tab.size(), one, L.team_resident)) return false;
    if (coarse && L.coarse.K > 4 * (int)tab.size()) return false;
    if (!one && !L.team_starts.now()) return false;
    TeamArgs T;
    T.K = coarse ? L.coarse.K : 0;
    T.ncd = L.coarse.ncd;
    T.nfree = L.coarse.nfree;
    T.lda = L.coarse.lda;
    if (T.K && (T.ncd > TEAM_VALUES || T.K > TEAM_TASKS)) return false;
    T.tab = B == 1 ? nullptr : L.team_tab.upload_get(tab.data(), tab.size(), s);
    T.vbeg = I.d_vbeg.p;
    bool cont = false;
    for (int i = 0; i < B; ++i) cont |= run[i] && L.h_it0[i];
    T.it0 = cont ? L.team_it0.upload_get(L.h_it0.data(), B, s) : nullptr;
    // published words; tags only grow, so words of earlier launches never match (cleared when they would wrap)
    const size_t n_pq = 2 * (size_t)A.nbA, n_r = 2 * (2 * (size_t)A.nbB + 8 * B), n_c = 2 * 7 * (size_t)T.K;
    const size_t nw = n_pq + n_r + n_c;
    const unsigned long long* had = L.team_words.p;
    unsigned long long* w = L.team_words.ensure(nw, s);
    if (w != had || L.team_tag > 0xffffffffull - (unsigned long long)A.maxit - 2) {
        IDP_LAUNCH(k_zero_words, grid_for((long)L.team_words.cap, 256), 256, 0, s, (long)L.team_words.cap, w);
        L.team_tag = 0;
    }
    T.w_pq = w;
    T.w_r = w + n_pq;
    T.w_rc = T.w_r + n_r;
    T.w_cp = T.w_rc + 12 * (size_t)T.K;
    T.tag0 = (unsigned)L.team_tag;
    L.team_tag += (unsigned long long)A.maxit + 2;
    T.ctl = team;
    T.done = team + 1;
    T.start = (unsigned*)(team + 1 + B);
    T.hand = team + 1 + 2 * B;
    T.start_limit = L.team_wait;
    T.nstart = handover ? nrun : 0;
    T.spin_limit = L.team_spin;
    T.aptr = L.coarse.aptr.p;
    T.avert = L.coarse.avert.p;
    T.Ps = L.coarse.Ps.p;
    T.Ainv = L.coarse.Ainv.p;
    static const void* const fns[] = {
        (const void*)k_pcg_team<false, false, false>, (const void*)k_pcg_team<false, true, false>,
        (const void*)k_pcg_team<false, false, true>,  (const void*)k_pcg_team<true, false, false>,
        (const void*)k_pcg_team<true, true, false>,   (const void*)k_pcg_team<true, false, true>};
    const void* fn = fns[(one ? 3 : 0) + (coarse ? 1 : handover ? 2 : 0)];
    PcgArgs a = A;
    void* args[] = {&a, &T};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    L.team_tok = L.prof ? L.prof->pair(e0, e1) : -1;
    if (e0) IDP_HIP(hipEventRecord(e0, s));
    IDP_HIP(hipLaunchKernel(fn, dim3(tab.size()), dim3(TEAM_THREADS), args, 0, s));
    if (e1) IDP_HIP(hipEventRecord(e1, s));
    return true;
}

// Preconditioned CG per instance on the assembled system (E + C); b, x: 3V.
// L.precond picks cluster (0: elastic and contact matching, 2: contact only) or 3x3 (1) block Jacobi.
// solve (device, B bytes; null = all) selects the instances to solve.
// Per instance on return: iters[i] >= 0, or -1 (singular diagonal block) /
// -2 (breakdown, p.q <= 0); relres[i] = |r|/|b|.
void pcg_solve_batch(LinWork& L, hipStream_t s, const MeshDev& m, const double* b, double* x, double rtol,
                     int maxit, const unsigned char* solve_h, int* iters, double* relres, const unsigned char* warm,
                     bool handover, bool one_kernel)
{
    const InstDev& I = m.inst;
    const int B = I.B;
    const int nV = m.nV;
    // per instance: 0 not solving, 1 new solve, 2 continued (its state is on the device)
    std::vector<unsigned char> sv(B, 1);
    if (solve_h) sv.assign(solve_h, solve_h + B);
    L.h_it0.resize(B, 0);
    L.h_maxit.assign(B, 0);
    for (int i = 0; i < B; ++i)
        if (sv[i] != 2) L.h_it0[i] = 0;
    // (null: the one solve of a plain mesh, a new one)
    const unsigned char* solve = B == 1 && sv[0] == 1 ? nullptr : L.solve_d.upload_get(sv.data(), B, s);
    const double nnzb = (double)m.nnzb_e + (double)L.ncb;
    // scalars, error and state flags and the team kernel's words (void mark,
    // iterations at a hand-over, start words, hand-over counts), in one piece:
    // they are read back together
    const int nteam = 1 + 2 * B + 2 * HAND_LOOKS + 1;
    const size_t nints = 2 * (size_t)B + 2 + nteam, nres = 3 * (size_t)B + 3;
    double* scal = L.scal.ensure(nres + (nints + 1) / 2, s);
    int* err = (int*)(scal + nres);
    int* flag = err + B;
    int* team = err + 2 * B + 2;
    IDP_LAUNCH(k_pcg_start, grid_for(std::max(B, nteam), 256), 256, 0, s, B, solve, flag, err, nteam, team);
    const bool haveC = L.ncb > 0;
    Profiler* P = L.prof;
    const int tok = P ? P->begin(IDP_K_PCG) : -1;
    // cluster block-Jacobi preconditioner
    const int vg = grid_for(nV, 256);
    int* best = L.cl_best.ensure(nV, s);
    int* root = L.cl_root.ensure(nV, s);
    int* size = L.cl_size.ensure(nV, s);
    int* root2 = L.cl_root2.ensure(nV, s);
    int* cnt = L.cl_cnt.ensure(nV, s);
    int* mem = L.cl_mem.ensure(CL_MAX * (size_t)nV, s);
    unsigned long long* pack = L.cl_pack.ensure(nV, s);
    double* Z = L.pinv.ensure(CL_ZS * (size_t)nV, s);
    int4* cm4 = (int4*)L.cl_cm4.ensure(4 * (size_t)nV, s);
    const int* crp = haveC ? L.crp.p : nullptr;
    const int* crp_match = L.precond != 1 ? crp : nullptr;  // no contact rows: singletons (3x3 block Jacobi)
    // precond 0: the matching weighs elastic couplings too, so clusters form
    // everywhere; precond 2: contact couplings only
    const ClElastic elm{L.precond == 0 ? m.e_rowptr.p : nullptr, m.e_col.p, L.evals.p, m.nnzb_e};
    // only the instances that solve (new or continued) build their clusters
    const ClMask cmk{I.vinst.p, solve};
    const int vgl = grid_for((long)CL_LANES * nV, 256);
    IDP_LAUNCH(k_cl_best, vgl, 256, 0, s, nV, crp_match, L.ccol.p, L.cvals.p, L.ncb, elm, cmk, best);
    IDP_LAUNCH(k_cl_pair, vg, 256, 0, s, nV, best, cmk, root, size);
    IDP_HIP(hipMemsetAsync(pack, 0, nV * sizeof(unsigned long long), s));
    IDP_LAUNCH(k_cl_best2, vgl, 256, 0, s, nV, crp_match, L.ccol.p, L.cvals.p, L.ncb, root, size, elm, cmk, pack);
    IDP_LAUNCH(k_cl_merge, vg, 256, 0, s, nV, root, pack, size, cmk, root2);
    IDP_HIP(hipMemsetAsync(cnt, 0, nV * sizeof(int), s));
    IDP_LAUNCH(k_cl_members, vg, 256, 0, s, nV, root2, cmk, cnt, mem);
    IDP_LAUNCH(k_cl_sort, vg, 256, 0, s, nV, root2, cnt, cmk, mem);
    IDP_LAUNCH(k_cl_build, grid_for(16L * nV, 256), 256, 0, s, nV, root2, cnt, mem, m.e_diag.p, m.e_rowptr.p, m.e_col.p, L.evals.p,
               m.nnzb_e, haveC ? L.cdiag.p : (const int*)nullptr, crp, L.ccol.p, L.cvals.p, L.ncb, I.vinst.p, cmk, Z,
               cm4, err);
    // coarse level: one instance with the positions of its system given
    const bool coarse = B == 1 && L.xpos && L.coarse.verts_per_agg > 0 && sv[0] == 1 && coarse_setup(L, s, m, L.xpos);
    PcgArgs A;
    A.nV = nV;
    A.cpart = coarse ? L.coarse.part.p : nullptr;
    A.cnsb = coarse ? L.coarse.nsb : 0;
    A.erp = m.e_rowptr.p;
    A.ecol = m.e_col.p;
    A.eval = L.evals.p;
    A.crp = haveC ? L.crp.p : nullptr;
    A.ccol = L.ccol.p;
    A.cval = L.cvals.p;
    A.eld = m.nnzb_e;
    A.cld = L.ncb;
    A.b = b;
    A.Z = Z;
    A.cm4 = cm4;
    A.x = x;
    A.r = L.r.ensure(6 * (size_t)nV, s);
    A.z = L.z.ensure(3 * (size_t)nV, s);
    A.pbuf = L.p.ensure(6 * (size_t)nV, s);
    A.q = L.q.ensure(3 * (size_t)nV, s);
    const SpmvShape shape = SPMV_SHAPES[L.spmv_shape];
    const int uw = std::min(std::max(L.upd_waves, 1), PCG_UPD_WAVES_MAX);
    const int gi = shape.g == 4 ? 0 : shape.g == 8 ? 1 : shape.g == 16 ? 2 : 3;
    const SegDev& rows = I.pcg_rows[gi];
    A.nbA = rows.nblk;
    A.nbB = I.pcg_upd.nblk;
    A.apbeg = rows.pbeg.p;
    A.bpbeg = I.pcg_upd.pbeg.p;
    // launch tables over the instances that solve (re-made as instances stop)
    std::vector<int> hf(2 * B);
    std::vector<char> run(B);
    for (int i = 0; i < B; ++i) run[i] = sv[i] != 0;  // as k_pcg_start sets the flags
    int nA = 0, nB = 0;
    double frac = 1.0;  // launched share of the rows (exact for one instance, row-proportional otherwise)
    auto tables = [&]() {
        if (B == 1 && run[0]) {  // one instance spans the launch: no table is read
            nA = A.nbA;
            nB = A.nbB;
            A.nbl_upd = nB;
            A.atab = A.btab = nullptr;
            A.aoff = A.boff = nullptr;
            A.ident = L.h_it0[0] + 1;  // iteration offset + 1
            return;
        }
        A.ident = 0;
        auto fill = [&](const SegDev& sd, std::vector<int4>& out, std::vector<int>& off) {
            out.clear();
            off.clear();
            for (int i = 0; i < B; ++i)
                if (run[i])
                    for (int k = sd.h_pbeg[i]; k < sd.h_pbeg[i + 1]; ++k) {
                        out.push_back(make_int4(sd.h_lo[k], sd.h_hi[k], i, k));
                        off.push_back(L.h_it0[i]);
                    }
        };
        fill(rows, L.h_atab, L.h_aoff);
        fill(I.pcg_upd, L.h_btab, L.h_boff);
        nA = (int)L.h_atab.size();
        nB = (int)L.h_btab.size();
        A.nbl_upd = nB;
        long rows = 0;
        for (const int4& t : L.h_btab) rows += t.y - t.x;
        frac = nV ? (double)rows / nV : 0.0;
        A.atab = L.atab.upload_get(L.h_atab.data(), L.h_atab.size(), s);
        A.btab = L.btab.upload_get(L.h_btab.data(), L.h_btab.size(), s);
        A.aoff = L.aoff.upload_get(L.h_aoff.data(), L.h_aoff.size(), s);
        A.boff = L.boff.upload_get(L.h_boff.data(), L.h_boff.size(), s);
    };
    A.solve = solve;
    tables();
    A.part_pq = L.part0.ensure(A.nbA + 1, s);
    A.part_bx = L.part_bx.ensure(A.nbA + 1, s);
    A.warm = warm;
    A.part_rz = L.part1.ensure(2 * (size_t)A.nbB + 2, s);
    A.part_rr = L.part2.ensure(2 * (size_t)A.nbB + 2, s);
    A.flag = flag;
    A.scal = scal;
    A.rtol2 = rtol * rtol;
    A.maxit = maxit;
    // one instance with many update blocks: reduce the partials once per
    // kernel boundary instead of in every block (IDP_PCG_PREREDUCE = 0 / 1
    // overrides the size rule)
    {
        const char* e = std::getenv("IDP_PCG_PREREDUCE");
        const int force = e ? std::atoi(e) : -1;
        const bool big = A.nbB >= PCG_PREREDUCE_BLOCKS;
        A.red = (B == 1 && A.ident && !coarse && (force < 0 ? big : force > 0)) ? L.red.ensure(8, s) : nullptr;
    }
    if (warm && nA) {
        if (shape.g == 4) IDP_LAUNCH(k_pcg_warm<4>, nA, PCG_ROW_THREADS, 0, s, A);
        else if (shape.g == 8) IDP_LAUNCH(k_pcg_warm<8>, nA, PCG_ROW_THREADS, 0, s, A);
        else if (shape.g == 16) IDP_LAUNCH(k_pcg_warm<16>, nA, PCG_ROW_THREADS, 0, s, A);
        else IDP_LAUNCH(k_pcg_warm<32>, nA, PCG_ROW_THREADS, 0, s, A);
    }
    auto spmv = [&](int it, hipEvent_t e0, hipEvent_t e1) {
        const int nt = PCG_ROW_THREADS + (shape.sw ? 64 : 0);
        switch (L.spmv_shape) {
        case 0: IDP_LAUNCH_TIMED((k_pcg_spmv<4, false>), nA, nt, 0, s, e0, e1, A, it); break;
        case 1: IDP_LAUNCH_TIMED((k_pcg_spmv<8, false>), nA, nt, 0, s, e0, e1, A, it); break;
        case 2: IDP_LAUNCH_TIMED((k_pcg_spmv<16, false>), nA, nt, 0, s, e0, e1, A, it); break;
        case 3: IDP_LAUNCH_TIMED((k_pcg_spmv<32, false>), nA, nt, 0, s, e0, e1, A, it); break;
        case 4: IDP_LAUNCH_TIMED((k_pcg_spmv<4, true>), nA, nt, 0, s, e0, e1, A, it); break;
        case 5: IDP_LAUNCH_TIMED((k_pcg_spmv<8, true>), nA, nt, 0, s, e0, e1, A, it); break;
        case 6: IDP_LAUNCH_TIMED((k_pcg_spmv<16, true>), nA, nt, 0, s, e0, e1, A, it); break;
        default: IDP_LAUNCH_TIMED((k_pcg_spmv<32, true>), nA, nt, 0, s, e0, e1, A, it); break;
        }
    };
    if (nB) IDP_LAUNCH(k_pcg_init, nB, PCG_UPD_BLOCK, 0, s, A);
    if (coarse) coarse_apply(L, s, nV, A.r, A.z, flag, 0);
    // algorithmic bytes of one SpMV launch (blocks + columns, two row-pointer
    // arrays, z and p_old read, p_new and q written) and of one update launch
    // (x, p, r, q, P^-1 read; x, r, z written)
    const double spmv_bytes = 76.0 * nnzb + 8.0 * (nV + 1) + 96.0 * nV;
    const double upd_bytes = 240.0 * nV;
    std::vector<double> hs(3 * B);
    // Hand-over (batched engine): once half of the new and continued solves
    // have stopped, the others get as many iterations again and then keep
    // their state for the next call.  One solve alone is never handed over.
    int nstart = 0;
    for (int i = 0; i < B; ++i) nstart += run[i];
    std::vector<int> hdone(B, 0), tstop(B, -1);  // one-kernel solves: handed over / stopped after these iterations
    bool teamed = one_kernel && nA > 0 && !(P && P->two_kernels()) && !A.red && shape.g == 8 &&
                  pcg_team(L, s, I, A, run, team, coarse, handover && nstart > 1);
    if (teamed) {
        double* h = L.pin->as<double>(nres + (nints + 1) / 2);
        IDP_HIP(hipMemcpyAsync(h, scal, (nres + (nints + 1) / 2) * sizeof(double), hipMemcpyDeviceToHost, s));
        IDP_HIP(hipStreamSynchronize(s));
        const int* hi = (const int*)(h + nres);
        if (hi[2 * B + 2]) {
            // a workgroup's wait for its team ran out: x and the vectors may be
            // half written, so every solve starts again, from zero
            if (P) P->end(IDP_K_PCG, tok);
            L.team_starts.ended(false);
            for (unsigned char& k : sv) k = k != 0;
            pcg_solve_batch(L, s, m, b, x, rtol, maxit, sv.data(), iters, relres, nullptr, handover, false);
            return;
        }
        std::copy(h, h + 3 * B, hs.begin());
        std::copy(hi, hi + 2 * B, hf.begin());
        bool left = false;
        for (int i = 0; i < B; ++i) {
            hdone[i] = hi[2 * B + 2 + 1 + i];
            if (run[i] && hf[B + i] != 0) tstop[i] = (int)hs[3 * i + 2] - L.h_it0[i];
            run[i] = run[i] && hf[B + i] == 0 && hdone[i] == 0;  // its team did not start
            left |= run[i] != 0;
        }
        L.team_starts.ended(!left);
        if (left) {
            teamed = false;
            tables();
        } else if (P) {
            P->end(IDP_K_PCG, tok);
        }
    }
    int it_half = -1, it_end = INT_MAX;
    int it = 0, chunk = 8;
    for (; !teamed && nA > 0 && it < it_end;) {
        for (int j = 0; j < chunk && it <= maxit && it < it_end; ++j, ++it) {
            // kernel times (events recorded by the dispatch itself) on one
            // iteration in 8
            const bool sample = P && (it & 7) == 3;
            hipEvent_t e0 = nullptr, e1 = nullptr;
            int t = sample ? P->pair(e0, e1) : -1;
            if (A.red) IDP_LAUNCH(k_pcg_red_spmv, 1, PCG_RED, 0, s, A, it);
            spmv(it, e0, e1);
            if (sample) P->end_pair(IDP_K_PCG_SPMV, t, spmv_bytes * frac, it);
            if (A.red) IDP_LAUNCH(k_pcg_red_upd, 1, PCG_RED, 0, s, A, it);
            t = sample ? P->pair(e0, e1) : -1;
            IDP_LAUNCH_TIMED(k_pcg_update, (nB + uw - 1) / uw, PCG_UPD_BLOCK * uw, 0, s, e0, e1, A, it);
            if (sample) P->end_pair(IDP_K_PCG_UPDATE, t, upd_bytes * frac, it);
            if (coarse) coarse_apply(L, s, nV, A.r + (size_t)((it + 1) & 1) * 3 * nV, A.z, flag, (it + 1) & 1);
        }
        IDP_HIP(hipMemcpyAsync(hf.data(), err, 2 * B * sizeof(int), hipMemcpyDeviceToHost, s));
        IDP_HIP(hipStreamSynchronize(s));
        bool fewer = false;
        int nrun = 0, later = 0;
        for (int i = 0; i < B; ++i) {
            if (run[i] && hf[B + i] != 0) {
                run[i] = 0;
                fewer = true;
            }
            nrun += run[i];
            later += tstop[i] >= it;  // stopped, in the one kernel, after more iterations
        }
        if (nrun == 0 || it > maxit) break;
        if (handover && nstart > 1 && it_half < 0 && 2 * (nrun + later) <= nstart) {
            it_half = it;
            it_end = 2 * it;
        }
        if (it >= it_end) break;
        if (fewer) tables();  // the stream is idle here: the tables may be rewritten
        chunk = std::min(chunk * 2, 256);
    }
    if (!teamed) {
        if (P) P->end(IDP_K_PCG, tok);
        IDP_HIP(hipMemcpyAsync(hs.data(), A.scal, 3 * B * sizeof(double), hipMemcpyDeviceToHost, s));
        IDP_HIP(hipStreamSynchronize(s));
    }
    int maxdone = 0;
    double done_iters = 0;
    for (int i = 0; i < B; ++i) {
        const int f = hf[B + i];
        iters[i] = 0;
        relres[i] = 0;
        if (f == 0) {
            const int did = hdone[i] ? hdone[i] : it;
            if (!hdone[i] && (teamed || it < it_end)) throw HipError(IDP_E_HIP, "PCG did not stop");
            iters[i] = PCG_HANDED_OVER;  // continues in the next call
            L.h_it0[i] += did;
            maxdone = std::max(maxdone, did);
            continue;
        }
        if (f == 3) continue;
        const int k = (int)hs[3 * i + 2];
        maxdone = std::max(maxdone, k - L.h_it0[i]);
        if (hf[i]) iters[i] = -1;
        else if (f == 2) iters[i] = -2;
        else {
            iters[i] = k;
            relres[i] = hs[3 * i] > 0 ? std::sqrt(hs[3 * i + 1] / hs[3 * i]) : 0.0;
            done_iters += k;
            if (f == 4) L.h_maxit[i] = 1;
        }
    }
    if (P) {
        if (teamed) {  // the whole solve as one launch: the bytes of all its iterations
            double w = 0.0;
            for (int i = 0; i < B; ++i) {
                const int k = hf[B + i] == 0 ? hdone[i] : hf[B + i] == 3 ? 0 : (int)hs[3 * i + 2] - L.h_it0[i];
                w += (spmv_bytes + upd_bytes) * k * (double)(I.vbeg[i + 1] - I.vbeg[i]) / std::max(nV, 1);
            }
            P->end_pair(IDP_K_PCG_SPMV, L.team_tok, w);
        }
        // launches at or after the last stopping iteration did no work
        P->discard_from(IDP_K_PCG_SPMV, maxdone);
        P->discard_from(IDP_K_PCG_UPDATE, maxdone);
        P->checkpoint();
        P->add_work(IDP_K_PCG, B == 1 ? done_iters * (spmv_bytes + upd_bytes) : 0.0);
    }
}

int pcg_solve_persistent(LinWork& L, hipStream_t s, const MeshDev& m, const double* b, double* x, double rtol,
                         int maxit, double* relres, const unsigned char* warm)
{
    int it = 0;
    double rel = 0;
    pcg_solve_batch(L, s, m, b, x, rtol, maxit, nullptr, &it, &rel, warm, false);
    *relres = rel;
    return it;
}

double dev_dot(LinWork& L, hipStream_t s, long n, const double* a, const double* b)
{
    int nblk = grid_for(n, RB);
    double* part = L.part3.ensure(nblk + 1, s);
    IDP_LAUNCH(k_dot_parts, nblk, RB, 0, s, n, a, b, part);
    IDP_LAUNCH(k_sum_partials, 1, RB, 0, s, nblk, part, part + nblk);
    double* v = L.pin->as<double>(1);
    IDP_HIP(hipMemcpyAsync(v, part + nblk, sizeof(double), hipMemcpyDeviceToHost, s));
    IDP_HIP(hipStreamSynchronize(s));
    return *v;
}

void dev_axpy(hipStream_t s, long n, const double* a, double sc, const double* b, double* x)
{
    IDP_LAUNCH(k_axpy3, grid_for(n, 256), 256, 0, s, n, a, sc, b, x);
}

void dev_velocity(hipStream_t s, long n, const double* x, const double* xn, double h, double* v)
{
    IDP_LAUNCH(k_velocity, grid_for(n, 256), 256, 0, s, n, x, xn, h, v);
}

void launch_sum_partials(hipStream_t s, int npart, const double* part, double* out)
{
    IDP_LAUNCH(k_sum_partials, 1, RB, 0, s, npart, part, out);
}

double dev_sum_partials(LinWork& L, hipStream_t s, int npart, const double* part)
{
    double* o = L.scal2.ensure(2, s);
    IDP_LAUNCH(k_sum_partials, 1, RB, 0, s, npart, part, o);
    double v;
    IDP_HIP(hipMemcpyAsync(&v, o, sizeof(double), hipMemcpyDeviceToHost, s));
    IDP_HIP(hipStreamSynchronize(s));
    return v;
}

}  // namespace idp
