// Newton linear solve on the device: H p = rhs for the system of the last assemble
// (NewtonLinearSystem::solve, CPU IPC/NewtonLinearSystem.cpp:21-56; tolerance and iteration
// cap as LinearSolverOptions.h:9-19, relative residual ||rhs - H p|| / ||rhs||).
//
// The matrix is used as a full symmetric 3x3-block matrix (BSR) built from the merged lower
// blocks of the assembly: every block (a, b), a > b, is also placed at (b, a) transposed.
// Zero entries that the CSR export drops contribute nothing to a product, so the two agree.
//
// Two precisions:
//   precision 0: FP64 conjugate gradients;
//   precision 1: the same iteration in FP32 (blocks, vectors) as the inner solver of FP64
//                iterative refinement: r = rhs - H x in FP64, solve H d = r in FP32, x += d,
//                until the FP64 residual meets the target.
// Three preconditioners: 3x3 block-Jacobi; a block lower-triangular factor G with
// M^-1 = G^T G, either the block FSAI of the matrix or the learned factor (learned.hip).
//
// Scalars (alpha, beta, norms) stay on the device and are combined from per-work-group
// partials in a fixed order (deterministic).  kCheck iterations are captured once into a
// HIP graph and replayed; the host checks convergence after each replay and kernels
// launched past convergence return at once.
#include <rocsolver/rocsolver.h>
#include "context.hpp"

#include <cmath>
#include <cstring>

namespace cipc {

constexpr int kPB = 256;       // threads per work-group (one vertex = 3 DOFs per thread)
constexpr int kCheck = 16;     // iterations between host convergence checks
constexpr int kMaxRefine = 64; // FP64 refinement steps of the mixed form

// device scalars of one solve
struct PcgScalars {
    double rz;        // r . z
    double rr;        // r . r
    double bn;        // ||b||
    double tol;       // absolute residual target
    double pq;        // p . q of the current iteration
    double beta;      // r.z' / r.z of the current iteration
    int done;         // converged (or broken down)
    int iters;
};

// ---- full symmetric BSR from the merged lower blocks -------------------------------
// The merged blocks k = (row a, column b), a >= b, are ordered by column, then row.  So the
// upper half of block row b, (b, a), is column b's run as it stands, and only the lower half
// of each row has to be found: counted per row, placed at its row by an atomic cursor, and
// ordered by rank (k ascends with the column).  With lowstart the scan of the lower counts,
// row i holds its lower entries at [lowstart[i] + mptr[i], ...), its diagonal at
// lowstart[i + 1] + mptr[i], and merged block k's upper entry is at lowstart[b + 1] + k.
// This takes the place of a radix sort of two mirrored 64-bit keys per block of capacity
// (merged blocks plus every empty record slot) and of three passes over the blocks (expand,
// convert, interleave): the set-up of a solve of four 20^3 cubes in contact
// (37,044 rows) 1.51 -> 1.23 ms with block FSAI and 0.70 -> 0.56 ms with block-Jacobi.
__global__ void bsr_count(int nm, const int* __restrict__ mrow, const int* __restrict__ mcol, const int* __restrict__ nm_ptr,
                          int* __restrict__ cnt) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nm || k >= *nm_ptr) return;
    const int a = mrow[k];
    if (a != mcol[k]) atomicAdd(cnt + a, 1);
}
__global__ void zero_i(int n, int* __restrict__ p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}
// the lower entries' merged blocks, at their row in any order (cnt counts back to zero); row
// starts and diagonal positions
__global__ void bsr_place(int nm, int V, const int* __restrict__ mrow, const int* __restrict__ mcol, const int* __restrict__ mptr,
                          const int* __restrict__ lowstart, int* __restrict__ cnt, int* __restrict__ low, int* __restrict__ rowptr,
                          int* __restrict__ dpos) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k <= V) rowptr[k] = lowstart[k] + mptr[k];
    if (k < V) dpos[k] = lowstart[k + 1] + mptr[k];
    if (k >= nm || k >= mptr[V]) return;
    const int a = mrow[k];
    if (a != mcol[k]) low[lowstart[a] + atomicSub(cnt + a, 1) - 1] = k;
}
// Interleaved layout of the blocks for the products: entries in groups of kGL, each group
// stored component-major (entry e, component k at (e / kGL) 9 kGL + k kGL + e % kGL), so that
// the kGL lanes of a row, which read consecutive entries, load each component with one
// contiguous access instead of nine 72-byte-strided ones.
constexpr int kGL = 8;         // lanes per block row of a product
__host__ __device__ inline size_t il_index(size_t e, int k) { return (e / kGL) * (9 * kGL) + (size_t)k * kGL + e % kGL; }
// Columns, mirror indices and blocks of both entries of every merged block.  A lane finds its
// block's two positions; the wavefront then writes its 64 blocks' components in merged order
// (coalesced reads).  vil / vilf: interleaved, val: plain 9-double blocks; null where unused.
__global__ __launch_bounds__(256) void bsr_fill(int nm, const int* __restrict__ mrow, const int* __restrict__ mcol,
                                                const int* __restrict__ nm_ptr, const double* __restrict__ mval,
                                                const int* __restrict__ lowstart, const int* __restrict__ low,
                                                const int* __restrict__ rowptr, int* __restrict__ col, int* __restrict__ mirror,
                                                double* __restrict__ vil, float* __restrict__ vilf, double* __restrict__ val) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63, k0 = k - lane;
    const int n = min(nm, *nm_ptr);
    if (k0 >= n) return;
    int up = -1, lo = -1;
    if (k < n) {
        const int a = mrow[k], b = mcol[k];
        up = lowstart[b + 1] + k;
        col[up] = a;
        if (a != b) {
            const int s0 = lowstart[a], s1 = lowstart[a + 1];
            lo = rowptr[a];
            for (int s = s0; s < s1; ++s) lo += low[s] < k;
            col[lo] = b;
            mirror[lo] = up;
            mirror[up] = lo;
        } else {
            mirror[up] = up;
        }
    }
    const int m = 9 * min(64, n - k0);
#pragma unroll
    for (int j = 0; j < 9; ++j) {
        const int t = 64 * j + lane, src = t / 9, c = t - 9 * src;
        const int u = __shfl(up, src), l = __shfl(lo, src);
        if (t >= m) continue;
        const double v = mval[(size_t)9 * k0 + t];
        const int ct = 3 * (c % 3) + c / 3;                   // (b, a) holds the transpose
        const int cu = l < 0 ? c : ct;                         // (the diagonal block as stored)
        if (vil) vil[il_index(u, cu)] = v;
        if (vilf) vilf[il_index(u, cu)] = (float)v;
        if (val) val[(size_t)9 * u + cu] = v;
        if (l >= 0) {
            if (vil) vil[il_index(l, c)] = v;
            if (vilf) vilf[il_index(l, c)] = (float)v;
            if (val) val[(size_t)9 * l + c] = v;
        }
    }
}
// block-Jacobi: inverse of each diagonal block (adjugate / determinant, symmetric), the
// block's values in the precision of the solve
template <typename T>
__global__ void diag_inverse(int V, const int* __restrict__ mptr, const int* __restrict__ mrow, const double* __restrict__ mval,
                             T* __restrict__ minv) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= V) return;
    double d[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    const int m = mptr[a];                                     // the first row of column a is a
    if (m < mptr[a + 1] && mrow[m] == a)
        for (int k = 0; k < 9; ++k) d[k] = (double)(T)mval[(size_t)9 * m + k];
    const double c00 = d[4] * d[8] - d[5] * d[7], c01 = d[5] * d[6] - d[3] * d[8], c02 = d[3] * d[7] - d[4] * d[6];
    const double det = d[0] * c00 + d[1] * c01 + d[2] * c02;
    const double id = det != 0.0 ? 1.0 / det : 0.0;
    const double inv[9] = {c00 * id, (d[2] * d[7] - d[1] * d[8]) * id, (d[1] * d[5] - d[2] * d[4]) * id,
                           c01 * id, (d[0] * d[8] - d[2] * d[6]) * id, (d[2] * d[3] - d[0] * d[5]) * id,
                           c02 * id, (d[1] * d[6] - d[0] * d[7]) * id, (d[0] * d[4] - d[1] * d[3]) * id};
    for (int k = 0; k < 9; ++k) minv[(size_t)9 * a + k] = (T)inv[k];
}

// ---- helpers ---------------------------------------------------------------------------
template <typename T>
__device__ inline void block_mv(const T* __restrict__ B, const T* __restrict__ x, double y[3]) {
    y[0] = (double)B[0] * x[0] + (double)B[1] * x[1] + (double)B[2] * x[2];
    y[1] = (double)B[3] * x[0] + (double)B[4] * x[1] + (double)B[5] * x[2];
    y[2] = (double)B[6] * x[0] + (double)B[7] * x[1] + (double)B[8] * x[2];
}
// Row-parallel sparse products: kGL lanes per 3x3-block row, so that the lanes of a row read
// consecutive blocks (coalesced), combined with cross-lane shuffles.  kRows rows per work-group.
constexpr int kRows = kPB / kGL;
template <typename T>
__device__ inline void group_reduce3(double y[3]) {
#pragma unroll
    for (int o = kGL / 2; o > 0; o >>= 1) {
        y[0] += __shfl_xor(y[0], o, kGL);
        y[1] += __shfl_xor(y[1], o, kGL);
        y[2] += __shfl_xor(y[2], o, kGL);
    }
}
template <typename T, typename X>
__device__ inline void block_mv_il(const T* __restrict__ B, size_t e, const X* __restrict__ x, double y[3]) {
    const T* b = B + (e / kGL) * (9 * kGL) + e % kGL;
    y[0] = (double)b[0] * x[0] + (double)b[kGL] * x[1] + (double)b[2 * kGL] * x[2];
    y[1] = (double)b[3 * kGL] * x[0] + (double)b[4 * kGL] * x[1] + (double)b[5 * kGL] * x[2];
    y[2] = (double)b[6 * kGL] * x[0] + (double)b[7 * kGL] * x[1] + (double)b[8 * kGL] * x[2];
}
// y = (A x)_a over entries rowptr[a] + sub, step kGL (all lanes of the group get the sum);
// val interleaved
template <typename T, typename X>
__device__ inline void row_product(int a, int sub, const int* __restrict__ rowptr, const int* __restrict__ col, const T* __restrict__ val,
                                   const X* __restrict__ x, double y[3]) {
    y[0] = y[1] = y[2] = 0.0;
    for (int e = rowptr[a] + sub; e < rowptr[a + 1]; e += kGL) {
        double t[3];
        block_mv_il(val, (size_t)e, x + 3 * (size_t)col[e], t);
        y[0] += t[0]; y[1] += t[1]; y[2] += t[2];
    }
    group_reduce3<T>(y);
}
// work-group sum of up to three values; thread 0 stores them at part[k * gridDim.x + blockIdx.x]
template <int K>
__device__ inline void group_partials(double v[K], double* __restrict__ part) {
    __shared__ double sh[K][kPB];
#pragma unroll
    for (int k = 0; k < K; ++k) sh[k][threadIdx.x] = v[k];
    __syncthreads();
    for (int s = kPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
#pragma unroll
            for (int k = 0; k < K; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) part[k * gridDim.x + blockIdx.x] = sh[k][0];
}
// work-group sums of two values stored to two partial arrays
__device__ inline void group_partials2(double v[2], double* __restrict__ pa, double* __restrict__ pb) {
    __shared__ double sh[2][kPB];
    sh[0][threadIdx.x] = v[0];
    sh[1][threadIdx.x] = v[1];
    __syncthreads();
    for (int s = kPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) { sh[0][threadIdx.x] += sh[0][threadIdx.x + s]; sh[1][threadIdx.x] += sh[1][threadIdx.x + s]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { pa[blockIdx.x] = sh[0][0]; pb[blockIdx.x] = sh[1][0]; }
}
// every work-group sums the partials of the previous kernel in the same order
__device__ inline double sum_partials_fixed(const double* __restrict__ part, int n) {
    __shared__ double sh[kPB];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += kPB) acc += part[i];
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    const double r = sh[0];
    __syncthreads();
    return r;
}

// ---- work-group layout of the row kernels ----------------------------------------------
// One system: work-group b covers block rows [b kRows, b kRows + kRows) of [0, V).  A batch of
// independent systems (block-diagonal matrix, one block per scene): bl[b] = {scene, first
// row, end row}; the work-groups of a scene are consecutive and never cover two scenes, and
// gb[k] .. gb[k + 1] are scene k's work-groups, so that the partials of one scene are summed
// exactly as those of the same system solved alone.
struct Layout {
    int V = 0, ng = 0;
    const int4* bl = nullptr;
    const int* gb = nullptr;
    __device__ void block(int& scene, int& row0, int& rend) const {
        if (bl) {
            const int4 t = bl[blockIdx.x];
            scene = t.x; row0 = t.y; rend = t.z;
        } else {
            scene = 0; row0 = blockIdx.x * kRows; rend = V;
        }
    }
    __device__ void parts(int scene, int& lo, int& n) const {
        if (gb) { lo = gb[scene]; n = gb[scene + 1] - lo; }
        else { lo = 0; n = ng; }
    }
};

// ---- PCG kernels (T: storage precision of blocks and vectors; scalars FP64) ------------
// Partials layout (ng work-groups each): [0] p.q, [1] r.z, [2] r.r, [3] b.b
// r = b - A x (A x skipped when x is zero); partials of r.r and b.b
// (grid: kRows block rows per work-group, kGL lanes per row)
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_residual(Layout L, const int* __restrict__ rowptr, const int* __restrict__ col,
                                                    const T* __restrict__ val, const double* __restrict__ b, const T* __restrict__ x,
                                                    int x_zero, T* __restrict__ r, double* __restrict__ part_rr,
                                                    double* __restrict__ part_bb) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double acc[2] = {0, 0};
    if (a < rend) {
        double y[3] = {0, 0, 0};
        if (!x_zero) row_product<T, T>(a, sub, rowptr, col, val, x, y);
        if (sub == 0) {
            const double rv[3] = {b[3 * a] - y[0], b[3 * a + 1] - y[1], b[3 * a + 2] - y[2]};
            acc[1] = b[3 * a] * b[3 * a] + b[3 * a + 1] * b[3 * a + 1] + b[3 * a + 2] * b[3 * a + 2];
            for (int k = 0; k < 3; ++k) r[3 * a + k] = (T)rv[k];
            acc[0] = (double)(T)rv[0] * (T)rv[0] + (double)(T)rv[1] * (T)rv[1] + (double)(T)rv[2] * (T)rv[2];
        }
    }
    group_partials2(acc, part_rr, part_bb);
}
// block-Jacobi: z = M^-1 r; partial of r.z; p = z when `init`
template <typename T>
__global__ __launch_bounds__(kPB) void prec_jacobi(Layout L, const T* __restrict__ minv, const T* __restrict__ r, T* __restrict__ z,
                                                   T* __restrict__ p, int init, const PcgScalars* __restrict__ sc,
                                                   double* __restrict__ part_rz) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    if (sc && sc[scene].done) return;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double acc[1] = {0.0};
    if (a < rend && sub == 0) {
        const T rt[3] = {r[3 * a], r[3 * a + 1], r[3 * a + 2]};
        double zv[3];
        block_mv(minv + (size_t)9 * a, rt, zv);
        for (int k = 0; k < 3; ++k) {
            z[3 * a + k] = (T)zv[k];
            if (init) p[3 * a + k] = (T)zv[k];
        }
        acc[0] = (double)rt[0] * (T)zv[0] + (double)rt[1] * (T)zv[1] + (double)rt[2] * (T)zv[2];
    }
    group_partials<1>(acc, part_rz);
}
// Factor preconditioner M^-1 = G^T G, G block lower-triangular.  F holds both products'
// blocks in the matrix's entry order, interleaved: entry (i, j) is G_ij for j <= i and G_ji^T
// above the diagonal, so that t = G r and z = G^T t both stream their half of each row (the
// transposed product used to gather 72-byte blocks through the mirror indices).
template <typename S, typename T>
__global__ void factor_entries(int V, const int* __restrict__ rowptr, const int* __restrict__ dpos, const int* __restrict__ mirror,
                               const S* __restrict__ G, T* __restrict__ F) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, a = t / kGL;
    if (a >= V) return;
    const int d = dpos[a], e1 = rowptr[a + 1];
    for (int e = rowptr[a] + t % kGL; e < e1; e += kGL) {
        const S* g = G + (size_t)9 * (e <= d ? e : mirror[e]);
        S v[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) v[k] = g[k];
#pragma unroll
        for (int k = 0; k < 9; ++k) F[il_index(e, k)] = (T)(e <= d ? v[k] : v[3 * (k % 3) + k / 3]);
    }
}
// row a's part of G r (entries up to the diagonal at d)
template <typename T, typename X>
__device__ inline void lower_product(int a, int sub, int e0, int d, const int* __restrict__ col, const T* __restrict__ F,
                                     const X* __restrict__ x, double y[3]) {
    y[0] = y[1] = y[2] = 0.0;
    for (int e = e0 + sub; e <= d; e += kGL) {
        double w[3];
        block_mv_il(F, (size_t)e, x + 3 * (size_t)col[e], w);
        y[0] += w[0]; y[1] += w[1]; y[2] += w[2];
    }
    group_reduce3<T>(y);
}
// row a's part of G^T t: the diagonal block transposed, the entries above it as stored
template <typename T, typename X>
__device__ inline void upper_product(int a, int sub, int d, int e1, const int* __restrict__ col, const T* __restrict__ F,
                                     const X* __restrict__ x, double y[3]) {
    y[0] = y[1] = y[2] = 0.0;
    for (int e = d + sub; e < e1; e += kGL) {
        const T* b = F + ((size_t)e / kGL) * (9 * kGL) + e % kGL;
        const X* xe = x + 3 * (size_t)col[e];
        const int s = e == d ? kGL : 3 * kGL, c = e == d ? 3 * kGL : kGL;   // row and column strides
        y[0] += (double)b[0] * xe[0] + (double)b[c] * xe[1] + (double)b[2 * c] * xe[2];
        y[1] += (double)b[s] * xe[0] + (double)b[s + c] * xe[1] + (double)b[s + 2 * c] * xe[2];
        y[2] += (double)b[2 * s] * xe[0] + (double)b[2 * s + c] * xe[1] + (double)b[2 * s + 2 * c] * xe[2];
    }
    group_reduce3<T>(y);
}
// t = G r
template <typename T>
__global__ __launch_bounds__(kPB) void prec_g1(Layout L, const int* __restrict__ rowptr, const int* __restrict__ dpos,
                                               const int* __restrict__ col, const T* __restrict__ F, const T* __restrict__ r,
                                               T* __restrict__ t, const PcgScalars* __restrict__ sc) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    if (sc && sc[scene].done) return;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    if (a >= rend) return;
    double y[3];
    lower_product(a, sub, rowptr[a], dpos[a], col, F, r, y);
    if (sub == 0)
        for (int k = 0; k < 3; ++k) t[3 * a + k] = (T)y[k];
}
// z = G^T t; partial of r.z; p = z when `init`
template <typename T>
__global__ __launch_bounds__(kPB) void prec_g2(Layout L, const int* __restrict__ rowptr, const int* __restrict__ dpos,
                                               const int* __restrict__ col, const T* __restrict__ F, const T* __restrict__ t,
                                               const T* __restrict__ r, T* __restrict__ z, T* __restrict__ p, int init,
                                               const PcgScalars* __restrict__ sc, double* __restrict__ part_rz) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    if (sc && sc[scene].done) return;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double acc[1] = {0.0};
    if (a < rend) {
        double y[3];
        upper_product(a, sub, dpos[a], rowptr[a + 1], col, F, t, y);
        if (sub == 0) {
            const T zt[3] = {(T)y[0], (T)y[1], (T)y[2]};
            for (int k = 0; k < 3; ++k) {
                z[3 * a + k] = zt[k];
                if (init) p[3 * a + k] = zt[k];
            }
            acc[0] = (double)r[3 * a] * zt[0] + (double)r[3 * a + 1] * zt[1] + (double)r[3 * a + 2] * zt[2];
        }
    }
    group_partials<1>(acc, part_rz);
}
// Per-scene controls of a batch solve (null for one system): relative tolerance, iteration
// cap and whether the scene takes part at all.
struct SceneControl {
    const double* rel_tol = nullptr;
    const int* max_iter = nullptr;
    const int* active = nullptr;
};
// scalars from the start partials: rz, rr, ||b|| (or ||r0|| as the reference of an inner
// solve); one work-group per scene
__global__ __launch_bounds__(kPB) void pcg_init_scalars(Layout L, const double* __restrict__ part_rz, const double* __restrict__ part_rr,
                                                        const double* __restrict__ part_bb, double rel_tol, int rel_to_r0,
                                                        SceneControl ctl, PcgScalars* __restrict__ sc) {
    const int k = blockIdx.x;
    int lo, n;
    L.parts(k, lo, n);
    const double rz = sum_partials_fixed(part_rz + lo, n);
    const double rr = sum_partials_fixed(part_rr + lo, n);
    const double bb = sum_partials_fixed(part_bb + lo, n);
    if (threadIdx.x == 0) {
        const double tol = ctl.rel_tol ? ctl.rel_tol[k] : rel_tol;
        PcgScalars& s = sc[k];
        s.rz = rz;
        s.rr = rr;
        s.bn = sqrt(bb);
        s.tol = tol * (rel_to_r0 ? sqrt(rr) : sqrt(bb));
        s.done = !(sqrt(rr) > s.tol) || !(rz > 0.0) || (ctl.active && !ctl.active[k]);
        s.iters = 0;
    }
}
// q = A p and partials of p.q
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_spmv(Layout L, const int* __restrict__ rowptr, const int* __restrict__ col,
                                                const T* __restrict__ val, const T* __restrict__ p, T* __restrict__ q,
                                                const PcgScalars* __restrict__ sc, double* __restrict__ part_pq) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    if (sc[scene].done) return;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double acc[1] = {0.0};
    if (a < rend) {
        double y[3];
        row_product<T, T>(a, sub, rowptr, col, val, p, y);
        if (sub == 0) {
            const T yt[3] = {(T)y[0], (T)y[1], (T)y[2]};
            for (int k = 0; k < 3; ++k) q[3 * a + k] = yt[k];
            acc[0] = (double)p[3 * a] * yt[0] + (double)p[3 * a + 1] * yt[1] + (double)p[3 * a + 2] * yt[2];
        }
    }
    group_partials<1>(acc, part_pq);
}
// p.q of every scene from the product's partials, once (one work-group per scene)
__global__ __launch_bounds__(kPB) void pcg_reduce_pq(Layout L, const double* __restrict__ part_pq, PcgScalars* __restrict__ sc) {
    const int k = blockIdx.x;
    if (sc[k].done) return;
    int lo, n;
    L.parts(k, lo, n);
    const double pq = sum_partials_fixed(part_pq + lo, n);
    if (threadIdx.x == 0) sc[k].pq = pq;
}
// alpha = rz / p.q; x += alpha p; r -= alpha q; partial of r.r; with block-Jacobi (minv set)
// also z = M^-1 r and its r.z partial
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_update(Layout L, const T* __restrict__ minv,
                                                  const T* __restrict__ p, const T* __restrict__ q, T* __restrict__ x, T* __restrict__ r,
                                                  T* __restrict__ z, const PcgScalars* __restrict__ sc, double* __restrict__ part_rz,
                                                  double* __restrict__ part_rr) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    if (sc[scene].done) return;
    const double alpha = sc[scene].rz / sc[scene].pq;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double acc[2] = {0.0, 0.0};
    if (a < rend && sub == 0) {
        T rt[3];
        for (int k = 0; k < 3; ++k) {
            x[3 * a + k] = (T)((double)x[3 * a + k] + alpha * (double)p[3 * a + k]);
            rt[k] = (T)((double)r[3 * a + k] - alpha * (double)q[3 * a + k]);
            r[3 * a + k] = rt[k];
        }
        if (minv) {
            double zv[3];
            block_mv(minv + (size_t)9 * a, rt, zv);
            for (int k = 0; k < 3; ++k) z[3 * a + k] = (T)zv[k];
            acc[0] = (double)rt[0] * (T)zv[0] + (double)rt[1] * (T)zv[1] + (double)rt[2] * (T)zv[2];
        }
        acc[1] = (double)rt[0] * rt[0] + (double)rt[1] * rt[1] + (double)rt[2] * rt[2];
    }
    if (minv) group_partials2(acc, part_rz, part_rr);
    else { double a1[1] = {acc[1]}; group_partials<1>(a1, part_rr); }
}
// p = z + beta p with the beta of pcg_scalars (one DOF per thread); skipped by a scene that
// has just converged, whose direction is no longer used
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_direction(int V, const T* __restrict__ z, T* __restrict__ p, const PcgScalars* __restrict__ sc) {
    if (sc->done) return;
    const double beta = sc->beta;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;       // one DOF per thread
    if (t < 3 * V) p[t] = (T)((double)z[t] + beta * (double)p[t]);
}
// the same on the row layout of a batch: the 3 kRows DOFs of the work-group's rows
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_direction_rows(Layout L, const T* __restrict__ z, T* __restrict__ p,
                                                          const PcgScalars* __restrict__ sc) {
    int scene, row0, rend;
    L.block(scene, row0, rend);
    if (sc[scene].done) return;
    const double beta = sc[scene].beta;
    const int t = 3 * row0 + threadIdx.x;
    if ((int)threadIdx.x < 3 * kRows && t < 3 * rend) p[t] = (T)((double)z[t] + beta * (double)p[t]);
}
// r.z', r.r and beta = r.z' / r.z from the partials, once per iteration (one work-group per
// scene); the convergence test
__global__ void pcg_scalars(Layout L, const double* __restrict__ part_rz, const double* __restrict__ part_rr,
                            PcgScalars* __restrict__ sc, int max_iter, SceneControl ctl) {
    const int k = blockIdx.x;
    if (sc[k].done) return;
    int lo, n;
    L.parts(k, lo, n);
    const double rz1 = sum_partials_fixed(part_rz + lo, n);
    const double rr = sum_partials_fixed(part_rr + lo, n);
    if (threadIdx.x == 0) {
        PcgScalars& s = sc[k];
        const int cap = ctl.max_iter ? ctl.max_iter[k] : max_iter;
        s.beta = rz1 / s.rz;
        s.rz = rz1;
        s.rr = rr;
        s.iters += 1;
        if (!(sqrt(rr) > s.tol) || s.iters >= cap || !(rz1 > 0.0)) s.done = 1;
    }
}
// x (FP64) += d (FP32), for the refinement (scenes with add[scene] != 0 when add is set)
__global__ void add_correction(int n, const float* __restrict__ d, double* __restrict__ x, const int* __restrict__ vs,
                               const int* __restrict__ add) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && (!add || add[vs[i / 3]])) x[i] += (double)d[i];
}
__global__ void zero_d(int n, double* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0.0;
}
__global__ void zero_f(int n, float* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0.0f;
}

// ---- block FSAI factor ----------------------------------------------------------------
// For block row i with lower pattern P (its entries j <= i, at most kFsaiMax blocks: the
// diagonal and the largest off-diagonal blocks by Frobenius norm), G_{i,P} is the last block
// row of L^-1, L the Cholesky factor of A[P,P]: then (G A G^T)_ii = I and G minimizes the
// Kaporin condition number over the pattern (Kolotilina & Yeremin's factorized sparse
// approximate inverse, in 3x3 blocks).  One wavefront per block row; A[P,P] in LDS.
//
// A row's cost is a chain of n dependent columns (a square root and a division each), so what
// counts is how many rows a CU has in flight and what a column costs.  M is packed by columns
// (no upper half: n (n + 1) / 2 doubles), which makes a column's reads over the lanes
// contiguous, and the factorisation is left-looking with lane = matrix row: two LDS reads and
// an FMA per element, no index arithmetic, no barrier (the work-group is one wavefront).  The
// LDS follows the row's size class: at most 10 blocks (3.7 KB; lattice interiors have 4 to 10,
// as many rows in flight as the wavefront slots allow), then 24 (21 KB) for the rows of
// vertices in contact, which the first launch lists for the second.  Solve set-up on
// the system of four 20^3 cubes in contact (37,044 rows) 4.34 -> 1.51 ms, of 24 scenes of up
// to 20^3 cells (80,390 rows) 7.96 -> 1.92 ms.
constexpr int kFsaiMax = 24;                   // blocks per row pattern
constexpr int kFsaiSmall = 10;                 // blocks per row of the first launch

__device__ inline int find_index(const int* __restrict__ a, int lo, int hi, int c) {
    while (lo < hi) { const int m = (lo + hi) >> 1; if (a[m] < c) lo = m + 1; else hi = m; }
    return lo;
}
// The matrix as the factor reads it: the BSR's pattern, the merged lower blocks' values.
struct FsaiMatrix {
    const int *rowptr, *dpos, *col, *mirror, *lowstart, *mptr, *mrow;
    const double* mval;
    // squared Frobenius norm of the block of lower entry e (its merged block follows from the
    // upper entry's position)
    __device__ double norm2(int e) const {
        const double* v = mval + (size_t)9 * (mirror[e] - lowstart[col[e] + 1]);
        double s = 0;
        for (int q = 0; q < 9; ++q) s += v[q] * v[q];
        return s;
    }
};
// (r, c), r >= c, of an n x n lower triangle packed by columns
__device__ inline int packed(int n, int c, int r) { return c * n - (c * (c - 1)) / 2 + (r - c); }

// One row, by one wavefront.  K: the most blocks of a row; rows with more go to big (their
// number in *nbig), K == kFsaiMax drops the smallest blocks instead.
template <int K>
__device__ inline void fsai_row(int i, const FsaiMatrix& A, double* __restrict__ G, double* __restrict__ M, int* __restrict__ P,
                                int* __restrict__ Pe, int* __restrict__ big, int* __restrict__ nbig) {
    const int lane = threadIdx.x;
    const int* __restrict__ col = A.col;
    const int e0 = A.rowptr[i], e1 = A.rowptr[i + 1];
    const int ediag = A.dpos[i];
    const int nl = ediag - e0;                            // off-diagonal lower candidates
    if (K < kFsaiMax && nl > K - 1) {
        if (lane == 0) big[atomicAdd(nbig, 1)] = i;
        return;
    }
    const bool all = nl <= K - 1;
    const int k = all ? nl + 1 : K;
    // the pattern's entries in column order, the diagonal last; the others' blocks are zero
    if (all) {
        for (int a = lane; a < k; a += 64) { Pe[a] = e0 + a; P[a] = col[e0 + a]; }
        for (size_t t = (size_t)9 * (ediag + 1) + lane; t < (size_t)9 * e1; t += 64) G[t] = 0.0;
    } else {
        // the K - 1 largest by Frobenius norm (ties by column)
        int kept = 0;
        for (int c0 = 0; c0 < nl; c0 += 64) {
            const int c = c0 + lane;
            bool keep = false;
            if (c < nl) {
                const double nc = A.norm2(e0 + c);
                int rank = 0;
                for (int o = 0; o < nl; ++o) {
                    const double no = A.norm2(e0 + o);
                    rank += (no > nc) || (no == nc && o < c);
                }
                keep = rank < K - 1;
            }
            const unsigned long long m = __ballot(keep);
            if (keep) {
                const int slot = kept + __popcll(m & ((1ull << lane) - 1));
                Pe[slot] = e0 + c;
                P[slot] = col[e0 + c];
            }
            kept += __popcll(m);
        }
        if (lane == 0) { Pe[K - 1] = ediag; P[K - 1] = i; }
        for (size_t t = (size_t)9 * e0 + lane; t < (size_t)9 * e1; t += 64) G[t] = 0.0;
    }
    __syncthreads();
    const int n = 3 * k;
    // M = A[P,P], lower triangle: blocks (a, b <= a) looked up in the merged columns of P
    for (int ab = lane; ab < k * (k + 1) / 2; ab += 64) {
        int a = (int)((sqrtf(8.0f * (float)ab + 1.0f) - 1.0f) * 0.5f);
        while ((a + 1) * (a + 2) / 2 <= ab) ++a;
        while (a * (a + 1) / 2 > ab) --a;
        const int b = ab - a * (a + 1) / 2;
        const int ce = A.mptr[P[b] + 1], f = find_index(A.mrow, A.mptr[P[b]], ce, P[a]);
        const bool has = f < ce && A.mrow[f] == P[a];
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
            for (int v = 0; v < 3; ++v)
                if (a != b || u >= v) M[packed(n, 3 * b + v, 3 * a + u)] = has ? A.mval[(size_t)9 * f + 3 * u + v] : 0.0;   // A_{P_a P_b}(u, v)
    }
    __syncthreads();
    // Cholesky M = L L^T, left-looking: lane r holds row r (and row 64 + r when 3 K > 64)
    constexpr int R = (3 * K + 63) / 64;
    for (int c = 0; c < n; ++c) {
        double s[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int r = lane + 64 * q;
            double s0 = 0.0, s1 = 0.0;
            if (r >= c && r < n) {
                s0 = M[packed(n, c, r)];
                int m = 0;
                for (; m + 1 < c; m += 2) {
                    const int b0 = packed(n, m, 0), b1 = packed(n, m + 1, 0);
                    s0 -= M[b0 + r] * M[b0 + c];
                    s1 -= M[b1 + r] * M[b1 + c];
                }
                if (m < c) { const int b0 = packed(n, m, 0); s0 -= M[b0 + r] * M[b0 + c]; }
            }
            s[q] = s0 + s1;
        }
        const double piv = R > 1 && c >= 64 ? __shfl(s[R - 1], c - 64) : __shfl(s[0], c);
        const double d = sqrt(fmax(piv, 1e-300));
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int r = lane + 64 * q;
            if (r == c) M[packed(n, c, r)] = d;
            else if (r > c && r < n) M[packed(n, c, r)] = s[q] / d;
        }
        __syncthreads();
    }
    // L^T Z = E (last three unit columns), from the last row up: lane r keeps row r of the
    // right-hand sides and subtracts L(s, r) z_s as each z_s is known
    double z[R][3];
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
        for (int u = 0; u < 3; ++u) z[q][u] = (lane + 64 * q == n - 3 + u) ? 1.0 : 0.0;
    for (int sr = n - 1; sr >= 0; --sr) {
        const double d = M[packed(n, sr, sr)];
        double zs[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) zs[u] = (R > 1 && sr >= 64 ? __shfl(z[R - 1][u], sr - 64) : __shfl(z[0][u], sr)) / d;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int r = lane + 64 * q;
            if (r == sr) {
#pragma unroll
                for (int u = 0; u < 3; ++u) z[q][u] = zs[u];
            } else if (r < sr) {
                const double l = M[packed(n, r, sr)];
#pragma unroll
                for (int u = 0; u < 3; ++u) z[q][u] -= l * zs[u];
            }
        }
    }
    // G_{i, P_a} (row u, column v) = Z[3a + v][u]
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int r = lane + 64 * q;
        if (r < n) {
            double* g = G + (size_t)9 * Pe[r / 3] + r % 3;
#pragma unroll
            for (int u = 0; u < 3; ++u) g[3 * u] = z[q][u];
        }
    }
    __syncthreads();   // the LDS is the next row's
}
// rows = null: the rows [0, V) of at most K blocks, the others listed; else the listed rows
template <int K>
__global__ __launch_bounds__(64) void fsai_rows(int V, const int* __restrict__ rows, int* __restrict__ nrows, FsaiMatrix A,
                                                double* __restrict__ G, int* __restrict__ big) {
    __shared__ double M[3 * K * (3 * K + 1) / 2];
    __shared__ int P[K], Pe[K];
    const int n = rows ? *nrows : V;
    for (int t = blockIdx.x; t < n; t += gridDim.x) fsai_row<K>(rows ? rows[t] : t, A, G, M, P, Pe, big, nrows);
}
// ---- host ---------------------------------------------------------------------------
namespace {
void read_scalars(Context& c, const PcgScalars* d, int S, std::vector<PcgScalars>& h) {
    h.resize(S);
    read_back(c, h.data(), d, (size_t)S);
}
bool all_done(const std::vector<PcgScalars>& h) {
    for (const PcgScalars& s : h)
        if (!s.done) return false;
    return true;
}

// The preconditioner of one solve: block-Jacobi (minv) or a factor (F, factor_entries).
template <typename T>
struct Prec {
    const T* minv = nullptr;
    const T* F = nullptr;
};

// Work-group layout of the current system: kRows block rows per work-group; for a batch
// the tables of per-scene work-groups (cached per vertex partition).
Layout make_layout(Context& c) {
    Scene& s = c.sc;
    SolveBuffers& w = c.solve;
    Layout L;
    L.V = s.V;
    if (s.S == 1) {
        L.ng = (int)blocks_for(s.V, kRows);
        return L;
    }
    if (w.layout_key != s.h_voff) {
        std::vector<int4> bl;
        std::vector<int> gb(s.S + 1, 0);
        for (int k = 0; k < s.S; ++k) {
            gb[k] = (int)bl.size();
            for (int r = s.h_voff[k]; r < s.h_voff[k + 1]; r += kRows) bl.push_back(make_int4(k, r, s.h_voff[k + 1], 0));
        }
        gb[s.S] = (int)bl.size();
        w.bl.resize(std::max<size_t>(bl.size(), 1));
        w.gb.resize(gb.size());
        CIPC_HIP(hipMemcpyAsync(w.bl.p, bl.data(), bl.size() * sizeof(int4), hipMemcpyHostToDevice, c.stream));
        CIPC_HIP(hipMemcpyAsync(w.gb.p, gb.data(), gb.size() * sizeof(int), hipMemcpyHostToDevice, c.stream));
        CIPC_HIP(hipStreamSynchronize(c.stream));
        w.layout_key = s.h_voff;
        w.layout_ng = (int)bl.size();
    }
    L.ng = w.layout_ng;
    L.bl = w.bl.p;
    L.gb = w.gb.p;
    return L;
}

template <typename T>
void apply_prec(Context& c, const Layout& L, const Prec<T>& M, const T* r, T* z, T* p, int init, const PcgScalars* sc, double* part_rz) {
    SolveBuffers& w = c.solve;
    if (M.F) {
        T* t = reinterpret_cast<T*>(w.t.p);
        hipLaunchKernelGGL(prec_g1<T>, dim3(L.ng), dim3(kPB), 0, c.stream, L, w.rowptr.p, w.dpos.p, w.col.p, M.F, r, t, sc);
        hipLaunchKernelGGL(prec_g2<T>, dim3(L.ng), dim3(kPB), 0, c.stream, L, w.rowptr.p, w.dpos.p, w.col.p, M.F, t, r, z, p, init, sc,
                           part_rz);
    } else {
        hipLaunchKernelGGL(prec_jacobi<T>, dim3(L.ng), dim3(kPB), 0, c.stream, L, M.minv, r, z, p, init, sc, part_rz);
    }
}

// PCG solves of A x = b (b FP64; A, x and the work vectors in T), one per scene in lock step.
// kCheck iterations are captured once into a HIP graph and replayed until the device flags
// say that every scene has converged.  Returns the scenes' final scalars.
template <typename T>
void pcg_run(Context& c, const Layout& L, int S, const T* val, const Prec<T>& M, const double* b, T* x, int x_zero, double rel_tol,
             int rel_to_r0, int max_iter, SceneControl ctl, std::vector<PcgScalars>& h) {
    const int V = c.sc.V;
    const int ng = L.ng;
    const int ngd = (int)blocks_for(3 * V, kPB);
    SolveBuffers& w = c.solve;
    T* r = reinterpret_cast<T*>(w.r.p);
    T* z = reinterpret_cast<T*>(w.z.p);
    T* p = reinterpret_cast<T*>(w.p.p);
    T* q = reinterpret_cast<T*>(w.q.p);
    double* part_pq = w.part.p;
    double* part_rz = w.part.p + ng;
    double* part_rr = w.part.p + 2 * ng;
    double* part_bb = w.part.p + 3 * ng;
    PcgScalars* sc = reinterpret_cast<PcgScalars*>(w.scal.p);
    hipLaunchKernelGGL(pcg_residual<T>, dim3(ng), dim3(kPB), 0, c.stream, L, w.rowptr.p, w.col.p, val, b, x, x_zero, r, part_rr, part_bb);
    apply_prec<T>(c, L, M, r, z, p, 1, nullptr, part_rz);
    hipLaunchKernelGGL(pcg_init_scalars, dim3(S), dim3(kPB), 0, c.stream, L, part_rz, part_rr, part_bb, rel_tol, rel_to_r0, ctl, sc);
    CIPC_CHECK_LAUNCH();
    read_scalars(c, sc, S, h);
    if (all_done(h)) return;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    CIPC_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < kCheck; ++k) {
        hipLaunchKernelGGL(pcg_spmv<T>, dim3(ng), dim3(kPB), 0, c.stream, L, w.rowptr.p, w.col.p, val, p, q, sc, part_pq);
        hipLaunchKernelGGL(pcg_reduce_pq, dim3(S), dim3(kPB), 0, c.stream, L, part_pq, sc);
        hipLaunchKernelGGL(pcg_update<T>, dim3(ng), dim3(kPB), 0, c.stream, L, M.F ? nullptr : M.minv, p, q, x, r, z, sc,
                           part_rz, part_rr);
        if (M.F) apply_prec<T>(c, L, M, r, z, p, 0, sc, part_rz);
        hipLaunchKernelGGL(pcg_scalars, dim3(S), dim3(kPB), 0, c.stream, L, part_rz, part_rr, sc, max_iter, ctl);
        if (L.bl) hipLaunchKernelGGL(pcg_direction_rows<T>, dim3(ng), dim3(kPB), 0, c.stream, L, z, p, sc);
        else hipLaunchKernelGGL(pcg_direction<T>, dim3(ngd), dim3(kPB), 0, c.stream, V, z, p, sc);
    }
    const hipError_t ce = hipStreamEndCapture(c.stream, &graph);
    CIPC_HIP(ce);
    CIPC_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    try {
        while (!all_done(h)) {
            CIPC_HIP(hipGraphLaunch(exec, c.stream));
            read_scalars(c, sc, S, h);
        }
    } catch (...) {
        (void)hipGraphExecDestroy(exec);
        (void)hipGraphDestroy(graph);
        throw;
    }
    (void)hipGraphExecDestroy(exec);
    (void)hipGraphDestroy(graph);
}

// Per-scene state of the FP64 refinement.
struct Refine {
    int iters = 0, outer = 0;
    bool finished = false;
    double rr = 0.0, bn = 0.0;
};
}  // namespace

// Full BSR of the last assembly: interleaved FP64 blocks and, for the mixed form, FP32; plain
// FP64 blocks when asked for (the learned factor's features).
void build_solve_matrix(Context& c, bool fp32, bool plain) {
    Scene& s = c.sc;
    const int V = s.V;
    SolveBuffers& w = c.solve;
    const size_t mcap = c.mrow.n;                 // merged blocks are bounded by the buffers' size
    const size_t ne = 2 * mcap, nil = (ne + kGL - 1) / kGL * 9 * kGL;
    w.low.resize(mcap); w.lowcnt.resize((size_t)V + 1); w.lowstart.resize((size_t)V + 1);
    w.col.resize(ne); w.mirror.resize(ne); w.rowptr.resize((size_t)V + 1); w.dpos.resize((size_t)V);
    w.vil.resize(nil);           // FP64: the solve, or the refinement's residuals
    if (fp32) w.vilf.resize(nil);
    if (plain) w.val.resize(9 * ne);
    const int* nm_ptr = c.mptr.p + V;
    const size_t np = std::max<size_t>(mcap, (size_t)V + 1);
    hipLaunchKernelGGL(zero_i, dim3(blocks_for((size_t)V + 1, 256)), dim3(256), 0, c.stream, V + 1, w.lowcnt.p);
    hipLaunchKernelGGL(bsr_count, dim3(blocks_for(mcap, 256)), dim3(256), 0, c.stream, (int)mcap, c.mrow.p, c.mcol.p, nm_ptr, w.lowcnt.p);
    CIPC_CHECK_LAUNCH();
    exclusive_scan_int(c, w.lowcnt.p, w.lowstart.p, V + 1);
    hipLaunchKernelGGL(bsr_place, dim3(blocks_for(np, 256)), dim3(256), 0, c.stream, (int)mcap, V, c.mrow.p, c.mcol.p, c.mptr.p,
                       w.lowstart.p, w.lowcnt.p, w.low.p, w.rowptr.p, w.dpos.p);
    hipLaunchKernelGGL(bsr_fill, dim3(blocks_for(mcap, 256)), dim3(256), 0, c.stream, (int)mcap, c.mrow.p, c.mcol.p, nm_ptr, c.mval.p,
                       w.lowstart.p, w.low.p, w.rowptr.p, w.col.p, w.mirror.p, w.vil.p, fp32 ? w.vilf.p : nullptr,
                       plain ? w.val.p : nullptr);
    CIPC_CHECK_LAUNCH();
    w.ne = ne;
}

// The block FSAI factor of the current BSR (plain blocks in w.G).
void build_fsai(Context& c) {
    SolveBuffers& w = c.solve;
    const int V = c.sc.V;
    w.G.resize(9 * w.ne);
    w.big.resize((size_t)V + 1);
    int* nbig = w.big.p + V;
    const FsaiMatrix A{w.rowptr.p, w.dpos.p, w.col.p, w.mirror.p, w.lowstart.p, c.mptr.p, c.mrow.p, c.mval.p};
    hipLaunchKernelGGL(zero_i, dim3(1), dim3(64), 0, c.stream, 1, nbig);
    hipLaunchKernelGGL(fsai_rows<kFsaiSmall>, dim3(V), dim3(64), 0, c.stream, V, (const int*)nullptr, nbig, A, w.G.p, w.big.p);
    hipLaunchKernelGGL(fsai_rows<kFsaiMax>, dim3(std::min(V, 256 * 7)), dim3(64), 0, c.stream, V, (const int*)w.big.p, nbig, A, w.G.p,
                       w.big.p);
    CIPC_CHECK_LAUNCH();
}

// One solve per scene of the last assembly (one scene: the plain solve).  Each scene runs
// the same iteration as it would alone: its own scalars, convergence test and refinement.
void linear_solve_scenes(Context& c, int precision, int preconditioner, double rel_tol, int max_iter, const int* active,
                         SolveResult* res) {
    Scene& s = c.sc;
    const int V = s.V, n = 3 * V, S = s.S;
    SolveBuffers& w = c.solve;
    const Layout L = make_layout(c);
    const int ng = L.ng;
    w.r.resize((size_t)n); w.z.resize((size_t)n); w.p.resize((size_t)n); w.q.resize((size_t)n); w.t.resize((size_t)n);
    w.part.resize((size_t)4 * ng);
    w.scal.resize((size_t)S * ((sizeof(PcgScalars) + 7) / 8));
    w.x.resize((size_t)n);
    const bool fp32 = precision == 1;
    build_solve_matrix(c, fp32, preconditioner == 2);
    w.factor = 0;
    Prec<double> Md;
    Prec<float> Mf;
    if (preconditioner == 0) {
        if (fp32) {
            w.minvf.resize((size_t)9 * V);
            hipLaunchKernelGGL(diag_inverse<float>, dim3(blocks_for(V, 256)), dim3(256), 0, c.stream, V, c.mptr.p, c.mrow.p, c.mval.p,
                               w.minvf.p);
        } else {
            w.minv.resize((size_t)9 * V);
            hipLaunchKernelGGL(diag_inverse<double>, dim3(blocks_for(V, 256)), dim3(256), 0, c.stream, V, c.mptr.p, c.mrow.p, c.mval.p,
                               w.minv.p);
        }
        Md.minv = w.minv.p; Mf.minv = w.minvf.p;
    } else {
        if (preconditioner == 1) build_fsai(c);
        else build_learned(c, fp32);
        const size_t nil = (w.ne + kGL - 1) / kGL * 9 * kGL;
        const dim3 grid(blocks_for((size_t)V * kGL, 256)), block(256);
        if (!fp32) {
            w.F.resize(nil);
            hipLaunchKernelGGL((factor_entries<double, double>), grid, block, 0, c.stream, V, w.rowptr.p, w.dpos.p, w.mirror.p, w.G.p, w.F.p);
        } else {
            w.Ff.resize(nil);
            if (preconditioner == 1)
                hipLaunchKernelGGL((factor_entries<double, float>), grid, block, 0, c.stream, V, w.rowptr.p, w.dpos.p, w.mirror.p, w.G.p,
                                   w.Ff.p);
            else
                hipLaunchKernelGGL((factor_entries<float, float>), grid, block, 0, c.stream, V, w.rowptr.p, w.dpos.p, w.mirror.p, w.Gf.p,
                                   w.Ff.p);
        }
        Md.F = w.F.p; Mf.F = w.Ff.p;
    }
    w.factor = preconditioner;
    CIPC_CHECK_LAUNCH();
    // per-scene controls (a batch): participation, inner tolerances and caps, correction mask
    SceneControl ctl;
    std::vector<int> act(S, 1);
    if (active)
        for (int k = 0; k < S; ++k) act[k] = active[k] ? 1 : 0;
    if (S > 1) {
        w.ctl_d.resize((size_t)S);
        w.ctl_i.resize(3 * (size_t)S);
        CIPC_HIP(hipMemcpyAsync(w.ctl_i.p, act.data(), S * sizeof(int), hipMemcpyHostToDevice, c.stream));
        ctl.active = w.ctl_i.p;
    }
    for (int k = 0; k < S; ++k) res[k] = SolveResult{};
    std::vector<PcgScalars> h;
    hipLaunchKernelGGL(zero_d, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, w.x.p);
    if (precision == 0) {
        pcg_run<double>(c, L, S, w.vil.p, Md, c.rhs.p, w.x.p, 1, rel_tol, 0, max_iter, ctl, h);
        for (int k = 0; k < S; ++k) {
            res[k].iterations = h[k].iters;
            res[k].rel_residual = h[k].bn > 0 ? std::sqrt(h[k].rr) / h[k].bn : 0.0;
        }
    } else {
        // FP64 refinement around FP32 PCG; each inner solve aims just past the remaining
        // reduction (floored at the FP32 reach), so one or two refinements usually suffice
        w.xf.resize((size_t)n); w.res.resize((size_t)n);
        double* part_rr = w.part.p + 2 * ng;
        double* part_bb = w.part.p + 3 * ng;
        PcgScalars* sc = reinterpret_cast<PcgScalars*>(w.scal.p);
        std::vector<Refine> st(S);
        for (int k = 0; k < S; ++k) st[k].finished = !act[k];
        std::vector<double> itol(S, 0.0);
        std::vector<int> icap(S, 0), need_inner(S, 0), add(S, 0);   // host sources of async copies: kept alive
        for (int round = 0;; ++round) {
            double* rd = w.res.p;
            hipLaunchKernelGGL(pcg_residual<double>, dim3(ng), dim3(kPB), 0, c.stream, L, w.rowptr.p, w.col.p, w.vil.p, c.rhs.p, w.x.p,
                               round == 0 ? 1 : 0, rd, part_rr, part_bb);
            hipLaunchKernelGGL(pcg_init_scalars, dim3(S), dim3(kPB), 0, c.stream, L, part_rr, part_rr, part_bb, rel_tol, 0, SceneControl{},
                               sc);
            CIPC_CHECK_LAUNCH();
            read_scalars(c, sc, S, h);
            bool any = false;
            for (int k = 0; k < S; ++k) {
                need_inner[k] = 0;
                if (st[k].finished) continue;
                st[k].rr = h[k].rr; st[k].bn = h[k].bn;
                if (!(std::sqrt(h[k].rr) > rel_tol * h[k].bn) || st[k].iters >= max_iter) { st[k].finished = true; continue; }
                const double need = rel_tol * h[k].bn / std::sqrt(h[k].rr);      // reduction still needed
                itol[k] = std::max(0.3 * need, 2e-6);
                icap[k] = max_iter - st[k].iters;
                need_inner[k] = 1;
                any = true;
            }
            if (!any) break;
            SceneControl ictl;
            if (S > 1) {
                CIPC_HIP(hipMemcpyAsync(w.ctl_d.p, itol.data(), S * sizeof(double), hipMemcpyHostToDevice, c.stream));
                CIPC_HIP(hipMemcpyAsync(w.ctl_i.p + S, icap.data(), S * sizeof(int), hipMemcpyHostToDevice, c.stream));
                CIPC_HIP(hipMemcpyAsync(w.ctl_i.p, need_inner.data(), S * sizeof(int), hipMemcpyHostToDevice, c.stream));
                ictl.rel_tol = w.ctl_d.p;
                ictl.max_iter = w.ctl_i.p + S;
                ictl.active = w.ctl_i.p;
            }
            hipLaunchKernelGGL(zero_f, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, w.xf.p);
            std::vector<PcgScalars> hi;
            pcg_run<float>(c, L, S, w.vilf.p, Mf, rd, w.xf.p, 1, itol[0], 1, icap[0], ictl, hi);
            // scenes that made no progress (breakdown) or hit the refinement cap stop here,
            // without their correction
            std::fill(add.begin(), add.end(), 0);
            for (int k = 0; k < S; ++k) {
                if (!need_inner[k]) continue;
                const int it = hi[k].iters;
                if (it == 0 || st[k].outer >= kMaxRefine) { st[k].finished = true; continue; }
                st[k].iters += it;
                ++st[k].outer;
                add[k] = 1;
            }
            if (S > 1) {
                CIPC_HIP(hipMemcpyAsync(w.ctl_i.p + 2 * S, add.data(), S * sizeof(int), hipMemcpyHostToDevice, c.stream));
                hipLaunchKernelGGL(add_correction, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, w.xf.p, w.x.p, s.vscene.p,
                                   w.ctl_i.p + 2 * S);
            } else if (add[0]) {
                hipLaunchKernelGGL(add_correction, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, w.xf.p, w.x.p, nullptr, nullptr);
            }
            CIPC_CHECK_LAUNCH();
        }
        for (int k = 0; k < S; ++k) {
            res[k].iterations = st[k].iters;
            res[k].refinements = st[k].outer;
            res[k].rel_residual = st[k].bn > 0 ? std::sqrt(st[k].rr) / st[k].bn : 0.0;
        }
    }
    // the Newton direction for the step bound and line search
    s.dir.resize((size_t)n);
    CIPC_HIP(hipMemcpyAsync(s.dir.p, w.x.p, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
    CIPC_HIP(hipStreamSynchronize(c.stream));
}

// ---- direct tier ------------------------------------------------------------------------
// The host direct solvers (PARDISO, CHOLMOD; NewtonLinearSystem.cpp:150-174) on the GPU: the
// assembled lower CSC scattered into a dense column-major matrix, factored by a dense
// Cholesky (rocSOLVER potrf) and solved (potrs); the FP64 residual of the solution is
// evaluated on the BSR as for PCG.  For systems up to kDirectMaxDofs unknowns.
__global__ void csc_lower_to_dense(int n, const int* __restrict__ outer, const int* __restrict__ inner, const double* __restrict__ val,
                                   double* __restrict__ A) {
    const int col = blockIdx.x * blockDim.x + threadIdx.x;
    if (col >= n) return;
    for (int k = outer[col]; k < outer[col + 1]; ++k) A[(size_t)col * n + inner[k]] = val[k];
}
__global__ void zero_dense(size_t n, double* __restrict__ A) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) A[i] = 0.0;
}

void direct_solve(Context& c, SolveResult& res) {
    Scene& s = c.sc;
    if (s.S != 1) throw Error(CIPC_ERR_LOGIC, "a batch is solved per scene");
    const int V = s.V, n = 3 * V;
    if (n > kDirectMaxDofs)
        throw Error(CIPC_ERR_INVALID_ARGUMENT, "the direct solve takes at most " + std::to_string(kDirectMaxDofs) + " unknowns, the system has " +
                                                   std::to_string(n));
    SolveBuffers& w = c.solve;
    w.dense.resize((size_t)n * n);
    w.x.resize((size_t)n);
    w.info.resize(1);
    if (!c.blas) {
        rocblas_handle h = nullptr;
        if (rocblas_create_handle(&h) != rocblas_status_success) throw Error(CIPC_ERR_HIP, "rocblas_create_handle failed");
        c.blas = h;
    }
    rocblas_handle h = static_cast<rocblas_handle>(c.blas);
    if (rocblas_set_stream(h, c.stream) != rocblas_status_success) throw Error(CIPC_ERR_HIP, "rocblas_set_stream failed");
    hipLaunchKernelGGL(zero_dense, dim3(4096), dim3(256), 0, c.stream, (size_t)n * n, w.dense.p);
    hipLaunchKernelGGL(csc_lower_to_dense, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, c.outer.p, c.inner.p, c.val.p, w.dense.p);
    CIPC_HIP(hipMemcpyAsync(w.x.p, c.rhs.p, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
    CIPC_CHECK_LAUNCH();
    if (rocsolver_dpotrf(h, rocblas_fill_lower, n, w.dense.p, n, w.info.p) != rocblas_status_success)
        throw Error(CIPC_ERR_HIP, "rocsolver_dpotrf failed");
    int info = 0;
    read_back(c, &info, w.info.p, 1);
    if (info != 0)
        throw Error(CIPC_ERR_RUNTIME, "the Newton system is not positive definite (Cholesky pivot " + std::to_string(info) + ")");
    if (rocsolver_dpotrs(h, rocblas_fill_lower, n, 1, w.dense.p, n, w.x.p, n) != rocblas_status_success)
        throw Error(CIPC_ERR_HIP, "rocsolver_dpotrs failed");
    // FP64 residual on the BSR of the same system
    build_solve_matrix(c, false, false);
    const Layout L = make_layout(c);
    const int ng = L.ng;
    w.r.resize((size_t)n);
    w.part.resize((size_t)4 * ng);
    w.scal.resize((sizeof(PcgScalars) + 7) / 8);
    double* part_rr = w.part.p + 2 * ng;
    double* part_bb = w.part.p + 3 * ng;
    PcgScalars* sc = reinterpret_cast<PcgScalars*>(w.scal.p);
    hipLaunchKernelGGL(pcg_residual<double>, dim3(ng), dim3(kPB), 0, c.stream, L, w.rowptr.p, w.col.p, w.vil.p, c.rhs.p, w.x.p, 0, w.r.p,
                       part_rr, part_bb);
    hipLaunchKernelGGL(pcg_init_scalars, dim3(1), dim3(kPB), 0, c.stream, L, part_rr, part_rr, part_bb, 1.0, 0, SceneControl{}, sc);
    CIPC_CHECK_LAUNCH();
    std::vector<PcgScalars> hs;
    read_scalars(c, sc, 1, hs);
    res.iterations = 0;
    res.refinements = 0;
    res.rel_residual = hs[0].bn > 0 ? std::sqrt(hs[0].rr) / hs[0].bn : 0.0;
    s.dir.resize((size_t)n);
    CIPC_HIP(hipMemcpyAsync(s.dir.p, w.x.p, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, c.stream));
    CIPC_HIP(hipStreamSynchronize(c.stream));
}

void destroy_direct(Context& c) {
    if (c.blas) (void)rocblas_destroy_handle(static_cast<rocblas_handle>(c.blas));
    c.blas = nullptr;
}

void linear_solve(Context& c, int precision, int preconditioner, double rel_tol, int max_iter, SolveResult& res) {
    if (c.sc.S != 1) throw Error(CIPC_ERR_LOGIC, "a batch is solved per scene");
    if (preconditioner == kDirectSolve) {
        direct_solve(c, res);
        return;
    }
    linear_solve_scenes(c, precision, preconditioner, rel_tol, max_iter, nullptr, &res);
}

}  // namespace cipc
