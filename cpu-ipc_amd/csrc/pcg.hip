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
// partials in a fixed order (deterministic).  An iteration is one launch per true dependency
// (pcg_product, pcg_update, pcg_factor); the host enqueues a few iterations ahead of the
// iteration number that the device reports through pinned memory, and launches that follow
// convergence return at once.
#include <rocsolver/rocsolver.h>
#include "context.hpp"
#include "lbvh.hpp"

#include <cmath>
#include <cstring>
#include <exception>

namespace cipc {

constexpr int kPB = 256;       // threads per work-group (one vertex = 3 DOFs per thread)
constexpr int kAhead = 6;      // iterations enqueued ahead of the device
constexpr int kOwnSums = 2048; // partials that every work-group adds up itself (pcg_sums otherwise)
constexpr int kMaxRefine = 64; // FP64 refinement steps of the mixed form

// device scalars of one solve
struct PcgScalars {
    double rz;        // r . z
    double rr;        // r . r
    double bn;        // ||b||
    double tol;       // absolute residual target
    int done;         // converged (or broken down)
    int iters;
};

// ---- full symmetric BSR from the merged lower blocks -------------------------------
// The merged blocks k = (row a, column b), a >= b, are ordered by column, then row.  So the
// upper half of block row b, (b, a), is column b's run as it stands, and only the lower half
// of each row has to be found: counted per row, placed at its row by an atomic cursor, and
// ordered by rank (k ascends with the column; each entry counts the smaller ones of its row, a
// loop over the row meant for the tens to hundreds of neighbours that meshes and contacts give:
// 91 us at 1,000, 831 at 10,000 and 3,290 at 40,000 neighbours of one vertex).  With lowstart the
// scan of the lower counts, row i holds its lower entries at [lowstart[i] + mptr[i], ...), its diagonal at
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
// Interleaved layout of the blocks for the products: entries in groups of kGL, a group's
// components 0..7 in 16-byte pieces (two doubles or four floats of one entry), piece by piece
// over the entries, then its components 8.  The kGL lanes of a row read consecutive entries, so
// each piece is one contiguous 128-byte access: five loads a block in FP64 and three in FP32,
// where component-major order took nine and 72-byte blocks nine strided ones.
constexpr int kGL = 8;         // lanes per block row of a product
template <typename T>
struct Wide;
template <>
struct Wide<double> { typedef double type __attribute__((ext_vector_type(2))); };
template <>
struct Wide<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <typename T>
__host__ __device__ inline size_t il_index(size_t e, int k) {
    constexpr int W = 16 / (int)sizeof(T);
    return (e / kGL) * (9 * kGL) + (k < 8 ? (size_t)(k / W) * (kGL * W) + (e % kGL) * W + k % W : 8 * kGL + e % kGL);
}
// the block of entry e, B its group's start
template <typename T>
__device__ inline void load_block(const T* __restrict__ B, unsigned e, T f[9]) {
    using V = typename Wide<T>::type;
    constexpr int W = 16 / (int)sizeof(T);
    const V* w = reinterpret_cast<const V*>(B) + e % kGL;
#pragma unroll
    for (int j = 0; j < 8 / W; ++j) {
        const V t = w[j * kGL];
#pragma unroll
        for (int i = 0; i < W; ++i) f[j * W + i] = t[i];
    }
    f[8] = B[8 * kGL + e % kGL];
}
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
        if (vil) vil[il_index<double>(u, cu)] = v;
        if (vilf) vilf[il_index<float>(u, cu)] = (float)v;
        if (val) val[(size_t)9 * u + cu] = v;
        if (l >= 0) {
            if (vil) vil[il_index<double>(l, c)] = v;
            if (vilf) vilf[il_index<float>(l, c)] = (float)v;
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
template <typename T>
__device__ inline void transpose3(T f[9]) {
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
        for (int m = 0; m < u; ++m) { const T w = f[3 * u + m]; f[3 * u + m] = f[3 * m + u]; f[3 * m + u] = w; }
}
// Row-parallel sparse products: kGL lanes per 3x3-block row, so that the lanes of a row read
// consecutive blocks (coalesced), combined with cross-lane shuffles.  kRows rows per work-group.
constexpr int kRows = kPB / kGL;
// v + v of the lane that the data-parallel-primitive control CTRL selects: the cross-lane sums
// go through the vector pipe (a few cycles a step) instead of LDS permutes (about a hundred)
template <int CTRL, int ROWS = 0xf>
__device__ inline double dpp_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140, kDppBcast15 = 0x142, kDppBcast31 = 0x143;
// sum over the kGL lanes of a row, in each of them
__device__ inline double row_sum(double v) { return dpp_add<kDppHalfMirror>(dpp_add<kDppXor2>(dpp_add<kDppXor1>(v))); }
// sum over the wavefront, in its last lane
__device__ inline double wave_sum(double v) {
    return dpp_add<kDppBcast31, 0xc>(dpp_add<kDppBcast15, 0xa>(dpp_add<kDppMirror>(row_sum(v))));
}
template <typename T>
__device__ inline void group_reduce3(double y[3]) {
#pragma unroll
    for (int u = 0; u < 3; ++u) y[u] = row_sum(y[u]);
}
template <typename T, typename X>
__device__ inline void block_mv_il(const T* __restrict__ B, size_t e, const X* __restrict__ x, double y[3]) {
    T f[9];
    load_block(B + (e / kGL) * (9 * kGL), (unsigned)e, f);
    block_mv(f, x, y);
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
// work-group sums of K values, the k-th stored at part[k][b]
template <int K>
__device__ inline void group_partials(int b, const double (&v)[K], double* const (&part)[K]) {
    __shared__ double sh[K][kPB / 64];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double s = wave_sum(v[k]);
        if ((threadIdx.x & 63) == 63) sh[k][threadIdx.x >> 6] = s;
    }
    __syncthreads();
    if (threadIdx.x < K) {
        double s = 0.0;
        for (int w = 0; w < kPB / 64; ++w) s += sh[threadIdx.x][w];
#pragma unroll
        for (int k = 0; k < K; ++k)
            if ((int)threadIdx.x == k) part[k][b] = s;
    }
}
// the sums of n partials of the previous kernel, in an order fixed by n, in every thread
template <int K>
__device__ inline void sum_partials_fixed(const double* const (&part)[K], int n, double (&out)[K]) {
    __shared__ double sh[K][kPB / 64];
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = 0.0;
    for (int i = threadIdx.x; i < n; i += kPB)
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] += part[k][i];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double s = wave_sum(out[k]);
        if ((threadIdx.x & 63) == 63) sh[k][threadIdx.x >> 6] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        out[k] = 0.0;
        for (int w = 0; w < kPB / 64; ++w) out[k] += sh[k][w];
    }
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
    // The work-group's place.  One system: each XCD takes a contiguous part of the rows, whose
    // neighbours mostly lie in the same part, so that its L2 holds an eighth of the vectors
    // and not all.  A batch stays round-robin: its scenes converge at different iterations, and
    // contiguous parts would leave XCDs without work (13.5 us against 10.8 us a product).
    __device__ int index() const { return bl ? (int)blockIdx.x : xcd_block(blockIdx.x, gridDim.x); }
    __device__ void block(int b, int& scene, int& row0, int& rend) const {
        if (bl) {
            const int4 t = bl[b];
            scene = t.x; row0 = t.y; rend = t.z;
        } else {
            scene = 0; row0 = b * kRows; rend = V;
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
    const int wg = L.index();
    int scene, row0, rend;
    L.block(wg, scene, row0, rend);
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
    group_partials<2>(wg, acc, {part_rr, part_bb});
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
        for (int k = 0; k < 9; ++k) F[il_index<T>(e, k)] = (T)(e <= d ? v[k] : v[3 * (k % 3) + k / 3]);
    }
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
    double v[3];
    sum_partials_fixed<3>({part_rz + lo, part_rr + lo, part_bb + lo}, n, v);
    if (threadIdx.x == 0) {
        const double tol = ctl.rel_tol ? ctl.rel_tol[k] : rel_tol;
        PcgScalars& s = sc[k];
        s.rz = v[0];
        s.rr = v[1];
        s.bn = sqrt(v[2]);
        s.tol = tol * (rel_to_r0 ? sqrt(v[1]) : sqrt(v[2]));
        s.done = !(sqrt(v[1]) > s.tol) || !(v[0] > 0.0) || (ctl.active && !ctl.active[k]);
        s.iters = 0;
    }
}

// One iteration is three launches with a factor and two with block-Jacobi, one per true
// dependency:
//   pcg_product  beta and the convergence test from the r.z and r.r partials; q = A p
//   pcg_update   alpha from the p.q partials; x += alpha p, r -= alpha q; t = G r or z = M^-1 r
//   pcg_factor   z = G^T t
// What used to be launches of their own is folded into these: the scalars are added up by every
// work-group from the partials (a scene of more than kOwnSums work-groups, where that read
// grows past the launch it saves, has pcg_sums do it), and a vector that a product gathers is
// combined where it is read, p = z + beta p_old and r = r_old - alpha q, so that no launch
// waits for the update.  Old and new p and r, and the scalars, therefore alternate between two
// buffers.  A vertex's z and p (and r and q) lie in one 8-component record and t in one of 4:
// a gather is three 16-byte loads in FP64 and two in FP32 where six 8- or 4-byte ones were,
// since what bounds these kernels is how many scattered lane loads a CU issues, not bytes.
// Against one launch per step, replayed as a graph of 16 iterations (us an iteration): four 20^3
// cubes in contact (37,044 rows) block FSAI 43.5 -> 34.3 FP64, 40 -> 25 FP32, block-Jacobi
// 28.9 -> 20.8; two 9^3 cubes (2,000 rows) block FSAI 18.5 -> 12.5, block-Jacobi 16.2 -> 8.9.
// Without the graph's capture a solve also starts sooner: block-Jacobi set-up 0.56 -> 0.12 ms.
// At 37,044 rows and FP64 the three take 10.8, 10.7 and 7.8 us (about 4 us each when empty):
// 34.6, 18.5 and 18.5 MB of blocks out of the last-level cache and the gathers' lane loads.
template <typename T>
struct PcgArgs {
    Layout L;
    int S, own_sums;
    const int *rowptr, *dpos, *col;
    const T *A, *F, *minv;
    const double* b;
    T *x, *zp[2], *rq[2], *t;
    double *part_pq, *part_rz, *part_rr, *part_bb, *sums;   // sums: 3 per scene, of pcg_sums
    PcgScalars* sc;                                         // two buffers of S
    int max_iter;
    SceneControl ctl;
    int* active;                                            // scenes not yet done
    volatile int* host;                                     // pinned: iterations begun, every scene done
};
// the two 3-vectors of an 8-component record, the one of a 4-component record
template <typename T>
__device__ inline void load_pair(const T* __restrict__ v, T a[3], T b[3]) {
    using V = typename Wide<T>::type;
    constexpr int W = 16 / (int)sizeof(T);
    T f[8];
#pragma unroll
    for (int j = 0; j < (W == 2 ? 3 : 2); ++j) {
        const V t = reinterpret_cast<const V*>(v)[j];
#pragma unroll
        for (int i = 0; i < W; ++i) f[j * W + i] = t[i];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) { a[i] = f[i]; b[i] = f[3 + i]; }
}
template <typename T>
__device__ inline void load_one(const T* __restrict__ v, T a[3]) {
    using V = typename Wide<T>::type;
    constexpr int W = 16 / (int)sizeof(T);
    const V t = *reinterpret_cast<const V*>(v);
    a[0] = t[0]; a[1] = t[1];
    if constexpr (W == 2) a[2] = v[2];
    else a[2] = t[2];
}
// Sum over entries e = s, s + kGL, ... < end of B_e v_e.  begin() puts the gathers and blocks of
// the first STEPS entries in flight (they need no scalar, so a kernel calls it before it adds
// up the partials), finish() multiplies and goes on, STEPS entries at a time.
template <typename T, int STEPS, typename Gather, typename Block>
struct RowProduct {
    typename Gather::raw v[STEPS];
    T f[STEPS][9];
    int s, end;
    __device__ void load(const Gather& gather, const Block& block) {
#pragma unroll
        for (int i = 0; i < STEPS; ++i)
            if (s + i * kGL < end) {
                gather.load(s + i * kGL, v[i]);
                block(s + i * kGL, f[i]);
            }
    }
    __device__ void begin(int first, int last, const Gather& gather, const Block& block) {
        s = first;
        end = last;
        load(gather, block);
    }
    __device__ void finish(const Gather& gather, const Block& block, double c, double y[3]) {
        y[0] = y[1] = y[2] = 0.0;
        while (s < end) {
#pragma unroll
            for (int i = 0; i < STEPS; ++i)
                if (s + i * kGL < end) {
                    T w[3];
                    gather.combine(v[i], c, w);
#pragma unroll
                    for (int u = 0; u < 3; ++u)
                        y[u] += (double)f[i][3 * u] * w[0] + (double)f[i][3 * u + 1] * w[1] + (double)f[i][3 * u + 2] * w[2];
                }
            s += STEPS * kGL;
            load(gather, block);
        }
#pragma unroll
        for (int u = 0; u < 3; ++u) y[u] = row_sum(y[u]);
    }
};
// interleaved blocks; with `transposed` >= 0 that entry's block transposed
template <typename T>
struct Blocks {
    const T* B;
    int transposed;
    __device__ void operator()(int e, T f[9]) const {
        load_block(B + (size_t)(e / kGL) * (9 * kGL), (unsigned)e, f);
        if (e == transposed) transpose3(f);
    }
};
// first + c second of a record, and the single vector
template <typename T>
struct PairGather {
    struct raw { T a[3], b[3]; };
    const T* v;
    const int* col;
    __device__ void load(int e, raw& r) const { load_pair(v + 8 * (size_t)col[e], r.a, r.b); }
    __device__ void combine(const raw& r, double c, T w[3]) const {
#pragma unroll
        for (int i = 0; i < 3; ++i) w[i] = (T)((double)r.a[i] + c * (double)r.b[i]);
    }
};
template <typename T>
struct OneGather {
    struct raw { T a[3]; };
    const T* v;
    const int* col;
    __device__ void load(int e, raw& r) const { load_one(v + 4 * (size_t)col[e], r.a); }
    __device__ void combine(const raw& r, double, T w[3]) const {
#pragma unroll
        for (int i = 0; i < 3; ++i) w[i] = r.a[i];
    }
};
template <typename T>
__device__ inline T pick3(int sub, const double y[3]) { return (T)(sub == 0 ? y[0] : sub == 1 ? y[1] : y[2]); }

// x = 0, r = b, q = p = 0 (the first direction is z + 0 p); partials of b.b; with block-Jacobi
// z and the r.z, r.r partials
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_start(PcgArgs<T> g) {
    const int wg = g.L.index();
    int scene, row0, rend;
    g.L.block(wg, scene, row0, rend);
    if (blockIdx.x == 0 && threadIdx.x == 0) *g.active = g.S;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double v[3] = {0, 0, 0};
    if (a < rend && sub < 3) {
        const double bv = g.b[3 * (size_t)a + sub];
        const T r = (T)bv;
        g.x[3 * (size_t)a + sub] = (T)0;
        g.rq[0][8 * (size_t)a + sub] = r;
        g.rq[0][8 * (size_t)a + 3 + sub] = (T)0;
        g.zp[0][8 * (size_t)a + 3 + sub] = (T)0;
        v[2] = bv * bv;
        if (g.minv) {
            const T* m = g.minv + 9 * (size_t)a + 3 * sub;
            const double* b = g.b + 3 * (size_t)a;
            const T z = (T)((double)m[0] * (T)b[0] + (double)m[1] * (T)b[1] + (double)m[2] * (T)b[2]);
            g.zp[0][8 * (size_t)a + sub] = z;
            v[0] = (double)r * z;
            v[1] = (double)r * r;
        }
    }
    group_partials<3>(wg, v, {g.part_rz, g.part_rr, g.part_bb});
}
// the scenes' sums of the previous launch's partials (K = 1: p.q; 2: r.z and r.r), one
// work-group per scene
template <int K>
__global__ __launch_bounds__(kPB) void pcg_sums(Layout L, const double* __restrict__ pa, const double* __restrict__ pb, double* __restrict__ sums) {
    int lo, n;
    L.parts(blockIdx.x, lo, n);
    double v[2] = {0, 0};
    if constexpr (K == 1) {
        double one[1];
        sum_partials_fixed<1>({pa + lo}, n, one);
        v[0] = one[0];
    } else {
        sum_partials_fixed<2>({pa + lo, pb + lo}, n, v);
    }
    if (threadIdx.x == 0)
        for (int k = 0; k < K; ++k) sums[3 * blockIdx.x + (K == 1 ? 0 : 1 + k)] = v[k];
}
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_product(PcgArgs<T> g, int it) {
    const int wg = g.L.index();
    int scene, row0, rend, lo, n;
    g.L.block(wg, scene, row0, rend);
    g.L.parts(scene, lo, n);
    const int cur = it & 1;
    PcgScalars s = g.sc[cur * g.S + scene];
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    const T* zp = g.zp[cur];
    const PairGather<T> gather{zp, g.col};
    const Blocks<T> block{g.A, -1};
    RowProduct<T, 2, PairGather<T>, Blocks<T>> prod;
    T z = (T)0, p = (T)0;
    if (!s.done && a < rend) {
        prod.begin(g.rowptr[a] + sub, g.rowptr[a + 1], gather, block);
        if (sub < 3) { z = zp[8 * (size_t)a + sub]; p = zp[8 * (size_t)a + 3 + sub]; }
    }
    bool ended = it == 0 && s.done;
    double beta = 0.0;
    if (it > 0 && !s.done) {
        double v[2];
        if (g.own_sums) sum_partials_fixed<2>({g.part_rz + lo, g.part_rr + lo}, n, v);
        else { v[0] = g.sums[3 * scene + 1]; v[1] = g.sums[3 * scene + 2]; }
        beta = v[0] / s.rz;
        s.rz = v[0];
        s.rr = v[1];
        s.iters += 1;
        const int cap = g.ctl.max_iter ? g.ctl.max_iter[scene] : g.max_iter;
        s.done = ended = !(sqrt(v[1]) > s.tol) || s.iters >= cap || !(v[0] > 0.0);
    }
    if (threadIdx.x == 0) {
        if (wg == lo) {
            g.sc[(cur ^ 1) * g.S + scene] = s;
            if (ended && atomicSub(g.active, 1) == 1) __hip_atomic_store(g.host + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (wg == 0) __hip_atomic_store(g.host, it + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (s.done) return;
    double acc[1] = {0.0};
    if (a < rend) {
        double y[3];
        prod.finish(gather, block, beta, y);
        if (sub < 3) {
            p = (T)((double)z + beta * (double)p);
            const T q = pick3<T>(sub, y);
            g.zp[cur ^ 1][8 * (size_t)a + 3 + sub] = p;
            g.rq[cur][8 * (size_t)a + 3 + sub] = q;
            acc[0] = (double)p * (double)q;
        }
    }
    group_partials<1>(wg, acc, {g.part_pq});
}
// it < 0: the start's t = G r
template <typename T, bool FACTOR>
__global__ __launch_bounds__(kPB) void pcg_update(PcgArgs<T> g, int it) {
    const int wg = g.L.index();
    int scene, row0, rend, lo, n;
    g.L.block(wg, scene, row0, rend);
    g.L.parts(scene, lo, n);
    const int cur = it < 0 ? 0 : it & 1;
    PcgScalars s;
    if (it >= 0) {
        s = g.sc[(cur ^ 1) * g.S + scene];
        if (s.done) return;
    }
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    const PairGather<T> gather{g.rq[cur], g.col};
    const Blocks<T> block{g.F, -1};
    RowProduct<T, 2, PairGather<T>, Blocks<T>> prod;
    T x = (T)0, p = (T)0, r = (T)0, q = (T)0, m[3] = {(T)0, (T)0, (T)0};
    if (a < rend) {
        if (FACTOR) prod.begin(g.rowptr[a] + sub, g.dpos[a] + 1, gather, block);
        if (it >= 0 && sub < 3) {
            const T* rq = g.rq[cur] + 8 * (size_t)a + sub;
            x = g.x[3 * (size_t)a + sub];
            p = g.zp[cur ^ 1][8 * (size_t)a + 3 + sub];
            r = rq[0];
            q = rq[3];
            if (!FACTOR)
#pragma unroll
                for (int i = 0; i < 3; ++i) m[i] = g.minv[9 * (size_t)a + 3 * sub + i];
        }
    }
    double alpha = 0.0;
    if (it >= 0) {
        double v[1];
        if (g.own_sums) sum_partials_fixed<1>({g.part_pq + lo}, n, v);
        else v[0] = g.sums[3 * scene];
        alpha = s.rz / v[0];
    }
    double acc[2] = {0.0, 0.0};
    if (a < rend) {
        if (it >= 0 && sub < 3) {
            g.x[3 * (size_t)a + sub] = (T)((double)x + alpha * (double)p);
            r = (T)((double)r - alpha * (double)q);
            g.rq[cur ^ 1][8 * (size_t)a + sub] = r;
        }
        if (FACTOR) {
            double y[3];
            prod.finish(gather, block, -alpha, y);
            if (sub < 3) g.t[4 * (size_t)a + sub] = pick3<T>(sub, y);
        } else {
            const T r0 = __shfl(r, 0, kGL), r1 = __shfl(r, 1, kGL), r2 = __shfl(r, 2, kGL);
            if (sub < 3) {
                const T z = (T)((double)m[0] * r0 + (double)m[1] * r1 + (double)m[2] * r2);
                g.zp[cur ^ 1][8 * (size_t)a + sub] = z;
                acc[0] = (double)r * (double)z;
                acc[1] = (double)r * (double)r;
            }
        }
    }
    if (!FACTOR) group_partials<2>(wg, acc, {g.part_rz, g.part_rr});
}
template <typename T>
__global__ __launch_bounds__(kPB) void pcg_factor(PcgArgs<T> g, int it) {
    const int wg = g.L.index();
    int scene, row0, rend;
    g.L.block(wg, scene, row0, rend);
    const int to = it < 0 ? 0 : (it & 1) ^ 1;
    if (it >= 0 && g.sc[to * g.S + scene].done) return;
    const int a = row0 + threadIdx.x / kGL, sub = threadIdx.x % kGL;
    double acc[2] = {0.0, 0.0};
    if (a < rend) {
        const int d = g.dpos[a];
        const OneGather<T> gather{g.t, g.col};
        const Blocks<T> block{g.F, d};   // the diagonal block is stored as G_aa
        RowProduct<T, 2, OneGather<T>, Blocks<T>> prod;
        prod.begin(d + sub, g.rowptr[a + 1], gather, block);
        const T r = sub < 3 ? g.rq[to][8 * (size_t)a + sub] : (T)0;
        double y[3];
        prod.finish(gather, block, 0.0, y);
        if (sub < 3) {
            const T z = pick3<T>(sub, y);
            g.zp[to][8 * (size_t)a + sub] = z;
            acc[0] = (double)r * (double)z;
            acc[1] = (double)r * (double)r;
        }
    }
    group_partials<2>(wg, acc, {g.part_rz, g.part_rr});
}
// x (FP64) += d (FP32), for the refinement (scenes with add[scene] != 0 when add is set)
__global__ void add_correction(int n, const float* __restrict__ d, double* __restrict__ x, const int* __restrict__ vs,
                               const int* __restrict__ add) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && (!add || add[vs[i / 3]])) x[i] += (double)d[i];
}
template <typename T>
__global__ void zero_v(int n, T* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = (T)0;
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

// PCG solves of A x = b from x = 0 (b FP64; A, x and the work vectors in T), one per scene in
// lock step.  The host keeps at most kAhead iterations enqueued beyond the one that the device
// last began, so that few launches follow the last scene's convergence.  Returns the scenes'
// final scalars.
template <typename T>
void pcg_run(Context& c, const Layout& L, int S, const T* val, const Prec<T>& M, const double* b, T* x, double rel_tol, int rel_to_r0,
             int max_iter, SceneControl ctl, std::vector<PcgScalars>& h) {
    const size_t V = (size_t)c.sc.V;
    SolveBuffers& w = c.solve;
    w.zp.resize(16 * V); w.rq.resize(16 * V); w.t.resize(4 * V);
    w.sums.resize(3 * (size_t)S);
    w.active.resize(1);
    c.pin_pcg.reserve(2);
    PcgArgs<T> g;
    g.L = L; g.S = S;
    int most = L.ng;
    if (S > 1) {
        most = 0;
        for (int k = 0; k < S; ++k) most = std::max(most, (int)blocks_for((size_t)(c.sc.h_voff[k + 1] - c.sc.h_voff[k]), kRows));
    }
    g.own_sums = most <= kOwnSums;
    g.rowptr = w.rowptr.p; g.dpos = w.dpos.p; g.col = w.col.p;
    g.A = val; g.F = M.F; g.minv = M.minv; g.b = b; g.x = x;
    for (int i = 0; i < 2; ++i) {
        g.zp[i] = reinterpret_cast<T*>(w.zp.p) + 8 * V * i;
        g.rq[i] = reinterpret_cast<T*>(w.rq.p) + 8 * V * i;
    }
    g.t = reinterpret_cast<T*>(w.t.p);
    g.part_pq = w.part.p; g.part_rz = w.part.p + L.ng; g.part_rr = w.part.p + 2 * (size_t)L.ng; g.part_bb = w.part.p + 3 * (size_t)L.ng;
    g.sums = w.sums.p;
    g.sc = reinterpret_cast<PcgScalars*>(w.scal.p);
    g.max_iter = max_iter; g.ctl = ctl;
    g.active = w.active.p;
    g.host = c.pin_pcg.p;
    volatile int* host = c.pin_pcg.p;
    host[0] = host[1] = 0;
    const dim3 rows(L.ng), threads(kPB);
    hipLaunchKernelGGL(pcg_start<T>, rows, threads, 0, c.stream, g);
    if (g.F) {
        hipLaunchKernelGGL((pcg_update<T, true>), rows, threads, 0, c.stream, g, -1);
        hipLaunchKernelGGL(pcg_factor<T>, rows, threads, 0, c.stream, g, -1);
    }
    hipLaunchKernelGGL(pcg_init_scalars, dim3(S), threads, 0, c.stream, L, g.part_rz, g.part_rr, g.part_bb, rel_tol, rel_to_r0, ctl, g.sc);
    CIPC_CHECK_LAUNCH();
    int it = 0;
    for (unsigned spins = 0; !host[1];) {
        if (it - host[0] >= kAhead) {
            // a failed launch or a lost device never reports: asked now and then
            if ((++spins & 0xfffff) == 0 && hipStreamQuery(c.stream) != hipErrorNotReady && it - host[0] >= kAhead && !host[1]) {
                CIPC_HIP(hipStreamSynchronize(c.stream));
                throw Error(CIPC_ERR_HIP, "the conjugate-gradient iteration stopped reporting");
            }
            continue;
        }
        hipLaunchKernelGGL(pcg_product<T>, rows, threads, 0, c.stream, g, it);
        if (!g.own_sums) hipLaunchKernelGGL(pcg_sums<1>, dim3(S), threads, 0, c.stream, L, g.part_pq, (const double*)nullptr, g.sums);
        if (g.F) {
            hipLaunchKernelGGL((pcg_update<T, true>), rows, threads, 0, c.stream, g, it);
            hipLaunchKernelGGL(pcg_factor<T>, rows, threads, 0, c.stream, g, it);
        } else {
            hipLaunchKernelGGL((pcg_update<T, false>), rows, threads, 0, c.stream, g, it);
        }
        if (!g.own_sums) hipLaunchKernelGGL(pcg_sums<2>, dim3(S), threads, 0, c.stream, L, g.part_rz, g.part_rr, g.sums);
        CIPC_CHECK_LAUNCH();
        ++it;
    }
    read_scalars(c, g.sc + (size_t)(it & 1) * S, S, h);
}

// Waits for the stream when a solve ends with an error: its iterations in flight still write the
// pinned progress words, which the next solve clears from the host and must find its own.
struct DrainOnError {
    Context& c;
    const int pending = std::uncaught_exceptions();
    ~DrainOnError() {
        if (std::uncaught_exceptions() > pending) (void)hipStreamSynchronize(c.stream);
    }
};

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
    const DrainOnError drain{c};
    const Layout L = make_layout(c);
    const int ng = L.ng;
    w.part.resize((size_t)4 * ng);
    w.scal.resize(2 * (size_t)S * ((sizeof(PcgScalars) + 7) / 8));
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
    if (precision == 0) {
        pcg_run<double>(c, L, S, w.vil.p, Md, c.rhs.p, w.x.p, rel_tol, 0, max_iter, ctl, h);
        for (int k = 0; k < S; ++k) {
            res[k].iterations = h[k].iters;
            res[k].rel_residual = h[k].bn > 0 ? std::sqrt(h[k].rr) / h[k].bn : 0.0;
        }
    } else {
        // FP64 refinement around FP32 PCG; each inner solve aims just past the remaining
        // reduction (floored at the FP32 reach), so one or two refinements usually suffice
        w.xf.resize((size_t)n); w.res.resize((size_t)n);
        hipLaunchKernelGGL(zero_v<double>, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, w.x.p);
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
            std::vector<PcgScalars> hi;
            pcg_run<float>(c, L, S, w.vilf.p, Mf, rd, w.xf.p, itol[0], 1, icap[0], ictl, hi);
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
