// Sparse assembly: contact records + static elastic blocks -> the reference's CSR.
//
// Reference: BHessian::toTriplets (CPU IPC/ContactMechanics.cpp:13-134) and
// NewtonLinearSystem::assemble (NewtonLinearSystem.cpp:126-154): lower-triangle entries
// (row >= col) of blocks whose two vertices are free, entries exactly equal to zero
// dropped before duplicates are summed, the mass diagonal on every DOF, Eigen's
// column-major lower storage (outer = column starts, inner = ascending rows), and the
// right-hand side zeroed on non-free vertices.
//
// Pipeline: contact records bucketed by block column (gradient records by vertex), each bucket
// ordered by rank and its equal blocks summed in record order by one work-group; the merged block
// and scalar entry counts of every column with the static pattern; one scan; one pass that writes
// the merged 3x3 blocks and the CSR, with exactly the scalar entries that received a nonzero
// contribution.
#include "context.hpp"

#include <hipcub/hipcub.hpp>

namespace cipc {

constexpr unsigned long long kNoKey = ~0ull;

void sort_u64(Context& c, const unsigned long long* kin, unsigned long long* kout, int n, int bits) {
    if (n <= 0) return;
    size_t bytes = 0;
    CIPC_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, bytes, kin, kout, n, 0, bits, c.stream));
    c.tmp.reserve(bytes);
    CIPC_HIP(hipcub::DeviceRadixSort::SortKeys(c.tmp.p, bytes, kin, kout, n, 0, bits, c.stream));
}
void sort_i32_pairs(Context& c, const int* kin, int* kout, const int* vin, int* vout, int n, int bits) {
    if (n <= 0) return;
    size_t bytes = 0;
    CIPC_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, kin, kout, vin, vout, n, 0, bits, c.stream));
    c.tmp.reserve(bytes);
    CIPC_HIP(hipcub::DeviceRadixSort::SortPairs(c.tmp.p, bytes, kin, kout, vin, vout, n, 0, bits, c.stream));
}
void sort_u32_pairs(Context& c, const unsigned* kin, unsigned* kout, const int* vin, int* vout, int n, int bits) {
    sort_u32_pairs(kin, kout, vin, vout, n, bits, c.stream, c.tmp);
}
void sort_u32_pairs(const unsigned* kin, unsigned* kout, const int* vin, int* vout, int n, int bits, hipStream_t st,
                    DBuf<unsigned char>& tmp) {
    if (n <= 0) return;
    size_t bytes = 0;
    CIPC_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, kin, kout, vin, vout, n, 0, bits, st));
    tmp.reserve(bytes);
    CIPC_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, kin, kout, vin, vout, n, 0, bits, st));
}
// out[i] = sum in[0..i-1]; out has n+1 entries when in has n (out[n] = total).
void exclusive_scan_int(Context& c, const int* in, int* out, int n) {
    size_t bytes = 0;
    CIPC_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, n, c.stream));
    c.tmp.reserve(bytes);
    CIPC_HIP(hipcub::DeviceScan::ExclusiveSum(c.tmp.p, bytes, in, out, n, c.stream));
}

// End of the run of `key` that starts at i in the sorted keys (galloping, then bisection), so
// that the summation loop has known bounds and its loads are independent.
template <typename K>
__device__ inline int run_end(const K* __restrict__ k, int n, int i, K key) {
    int a = i, b = i + 1, st = 1;
    while (b < n && k[b] == key) { a = b; st <<= 1; b = i + st; }
    if (b > n) b = n;
    while (b - a > 1) { const int m = (a + b) >> 1; if (k[m] == key) a = m; else b = m; }
    return b;
}
// --- contact gradient records, summed per vertex in record order ------------------
__global__ void add_gradient_records(int n, const int* __restrict__ k, const int* __restrict__ idx,
                                     const double* __restrict__ val, int V, double* __restrict__ grad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int v = k[i];
    if (v < 0 || v >= V || (i > 0 && k[i - 1] == v)) return;
    const int e = run_end(k, n, i, v);
    double g0 = grad[3 * v], g1 = grad[3 * v + 1], g2 = grad[3 * v + 2];
#pragma unroll 2
    for (int j = i; j < e; ++j) {
        const double* p = val + (size_t)3 * idx[j];
        g0 += p[0]; g1 += p[1]; g2 += p[2];
    }
    grad[3 * v] = g0; grad[3 * v + 1] = g1; grad[3 * v + 2] = g2;
}
void add_gradient_records_into(Context& c, int n, const int* k, const int* idx, const double* val, double* grad) {
    if (n <= 0) return;
    hipLaunchKernelGGL(add_gradient_records, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, k, idx, val, c.sc.V, grad);
    CIPC_CHECK_LAUNCH();
}
// --- static and contact blocks merged per block column; the scalar CSR -------------------
// A block's flags: bit 3r + c set where entry (r, c) received a nonzero contribution.  Scalar
// column 3b + c lists, for each merged block of block column b in row order, the rows r of the
// block with a flag at (r, c) (r >= c on the diagonal block).
constexpr unsigned kLowerFlags = 0x1d9u;   // (r, c) with r >= c
__device__ inline unsigned csr_flags(unsigned f, bool diagonal) { return diagonal ? f & kLowerFlags : f; }

struct Merge {
    int V, nblocks, nb;
    const int *scol, *srow;              // static blocks
    const double* sbv;
    const unsigned short* sbf;
    int* ucnt;                           // unique contact blocks of column b: ucnt[2b], at ustart[2b]
    const int *ustart, *urow;
    const double* uval;
    const unsigned short* uflag;
    const int* mstart;
    int2* src;                           // (static, contact) block or -1 of each merged block, at mstart
    int *count, *off;                    // merged blocks per column (V + 1), then entries per scalar column (3V + 1)
    int* totals;
    const int* bt;
    const double* grad;
    int *mrow, *mcol;
    double* mval;
    int *outer, *inner, *nnz_out;
    double *val, *rhs;
};
// One thread per block column: how many blocks and scalar entries it has, and, where it has
// contact blocks, which two each merged block comes from.  Only flags and rows are read: the
// values wait for csr_fill, which knows every start.
__global__ void merge_count(Merge a) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    int* entries = a.count + a.V + 1;
    if (b == 0) {   // the scan's tails
        a.count[a.V] = 0;
        entries[3 * a.V] = 0;
    }
    if (b >= a.V) return;
    const int nu = a.ucnt[2 * b], ie = a.scol[b + 1];
    int i = a.scol[b], n = 0, e0 = 0, e1 = 0, e2 = 0;
    auto add = [&](unsigned f) {
        ++n;
        e0 += __popc(f & 0x49u);
        e1 += __popc(f & 0x92u);
        e2 += __popc(f & 0x124u);
    };
    if (nu == 0) {
        for (; i < ie; ++i) add(csr_flags(a.sbf[i], a.srow[i] == b));
    } else {
        int j = a.ustart[2 * b];
        const int je = j + nu;
        int2* src = a.src + a.mstart[b];
        while (i < ie || j < je) {
            const int ra = i < ie ? a.srow[i] : 0x7fffffff, rb = j < je ? a.urow[j] : 0x7fffffff;
            const bool st = ra <= rb, co = rb <= ra;
            src[n] = make_int2(st ? i : -1, co ? j : -1);
            add(csr_flags((st ? a.sbf[i] : 0u) | (co ? a.uflag[j] : 0u), min(ra, rb) == b));
            i += st ? 1 : 0;
            j += co ? 1 : 0;
        }
    }
    a.count[b] = n;
    entries[3 * b] = e0; entries[3 * b + 1] = e1; entries[3 * b + 2] = e2;
}
// The merged blocks, the CSR and the right-hand side in one pass: kFillLanes lanes per block
// column, a merged block each (most columns have 7 or 8).  A lane's scalar entries follow those
// of the lanes before it, which ballots count.  It is bound by its stores (a 72-byte block is
// written twice, once with its indices): 94 us on four 32^3 cubes (1.1 million blocks), where a
// thread per column, counts per block and component, their scan and a fill took 205.
constexpr int kFillLanes = 8;
__global__ __launch_bounds__(256) void csr_fill(Merge a) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int b = t / kFillLanes, l = t % kFillLanes, g0 = (threadIdx.x & 63) - l;
    const int base = a.off[a.V + 1];   // the entries' counts follow the blocks' in the scan
    const int* ent = a.off + a.V + 1;
    if (t == 0) {
        const int nnz = ent[3 * a.V] - base;
        a.outer[3 * a.V] = nnz;
        *a.nnz_out = nnz;
        a.totals[0] = a.totals[1] = a.totals[2] = a.totals[3] = 0;   // the buckets' totals for the next assembly
    }
    const bool on = b < a.V;
    int m0 = 0, nm = 0, nu = 0, s0 = 0;
    int pos[3] = {0, 0, 0};
    const int2* src = nullptr;
    if (on) {
        m0 = a.off[b];
        nm = a.off[b + 1] - m0;
        nu = a.ucnt[2 * b];
        s0 = a.scol[b];
        if (nu) src = a.src + a.mstart[b];
        for (int c = 0; c < 3; ++c) pos[c] = ent[3 * b + c] - base;
        if (l < 3) {
            a.outer[3 * b + l] = l == 0 ? pos[0] : l == 1 ? pos[1] : pos[2];
            a.rhs[3 * (size_t)b + l] = is_free(a.bt[b]) ? a.grad[3 * (size_t)b + l] : 0.0;
        }
    }
    const unsigned long long before = (1ull << l) - 1, lanes = (1ull << kFillLanes) - 1;
    for (int p0 = 0; __any(p0 < nm); p0 += kFillLanes) {
        const int p = p0 + l;
        const bool has = p < nm;
        int i = -1, j = -1, row = 0;
        unsigned f = 0;
        double v[9];
        if (has) {
            if (nu) {
                const int2 x = src[p];
                i = x.x; j = x.y;
            } else {
                i = s0 + p;
            }
            row = i >= 0 ? a.srow[i] : a.urow[j];
            if (i >= 0) {
                f = a.sbf[i];
#pragma unroll
                for (int e = 0; e < 9; ++e) v[e] = a.sbv[(size_t)9 * i + e];
            } else {
#pragma unroll
                for (int e = 0; e < 9; ++e) v[e] = 0.0;
            }
            if (j >= 0) {
                f |= a.uflag[j];
#pragma unroll
                for (int e = 0; e < 9; ++e) v[e] += a.uval[(size_t)9 * j + e];
            }
            const size_t o = (size_t)m0 + p;
            a.mrow[o] = row;
            a.mcol[o] = b;
#pragma unroll
            for (int e = 0; e < 9; ++e) a.mval[9 * o + e] = v[e];
            f = csr_flags(f, row == b);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            int o = pos[c], all = 0;
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const unsigned long long m = (__ballot((f >> (3 * r + c)) & 1u) >> g0) & lanes;
                o += __popcll(m & before);
                all += __popcll(m);
            }
#pragma unroll
            for (int r = 0; r < 3; ++r)
                if ((f >> (3 * r + c)) & 1u) {
                    a.inner[o] = 3 * row + r;
                    a.val[o] = v[3 * r + c];
                    ++o;
                }
            pos[c] += all;
        }
    }
    if (on && l == 0 && nu) a.ucnt[2 * b] = 0;   // for the next assembly's bucket counts
}

// Collision count as compute_g_dpt returns it (ContactMechanics.cpp:2970-3032): the
// multiplicity of a point-point / point-edge entry, one for every other Self_ActiveSet entry.
// out[1] = the count, out[0] = the CSR's nonzeros (csr_fill): read by the host together.  The
// work-groups add their sums to out[2], and the last of them (out[3] counts) publishes and
// clears both.  (One work-group over the whole set took 336 us on a folded 128^2 cloth's 105,000
// entries, 9 now.)
constexpr int kCountGroups = 128;
__global__ __launch_bounds__(256) void collision_count(const int* __restrict__ n_dev, const int4* __restrict__ set, int* out) {
    __shared__ int sh[4];
    int acc = 0;
    const int n = *n_dev;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const int4 e = set[i];
        acc += (e.x < 0 && (e.z < 0 || e.w < 0)) ? -e.w : 1;
    }
    for (int w = 32; w > 0; w >>= 1) acc += __shfl_xor(acc, w);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x != 0) return;
    acc = sh[0] + sh[1] + sh[2] + sh[3];
    atomicAdd(out + 2, acc);
    __threadfence();
    if (atomicAdd(out + 3, 1) == (int)gridDim.x - 1) {
        __threadfence();
        out[1] = atomicExch(out + 2, 0);
        atomicExch(out + 3, 0);
    }
}

__global__ void zero_ints(int* __restrict__ p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// --- contact records bucketed by vertex and summed --------------------------------------
// Bucket 2v holds the block records of block column v, bucket 2v + 1 the gradient records of
// vertex v.  The kernels that write the records count them (Records in contact.hip: one atomic
// per contact and vertex gives the records of both buckets their slots).  Then a start per
// bucket that has records, from running totals (where a bucket lies decides nothing), and the
// list of those buckets; the scatter; and one work-group per listed bucket that puts its records
// in the order of a stable sort by key and sums them in that order.  Most vertices of a body are
// in no contact, so nothing is launched per vertex but the pass over the counts.
struct Buckets {
    int V, kb, nb, ng;
    const unsigned long long* bkey;
    const int *gkey, *slot;           // slot: nb block records', then ng gradient records'
    int *cnt, *start, *list;          // 2V
    int* mstart;                      // V: room for a column's merged blocks
    const int* scol;
    int* totals;                      // listed buckets, block entries, gradient entries, merged blocks of columns with entries
    unsigned long long *entries, *sorted;   // nb + ng: (row, record) of blocks, then records of gradients
    const double *cval, *gval;
    int* urow;                        // at a column's start: its unique blocks
    double* uval;
    unsigned short* uflag;
    double* grad;
};
__device__ inline int wave_prefix(int v, int& total) {
    const int lane = threadIdx.x & 63;
    int x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    total = __shfl(x, 63);
    return x - v;
}
// One atomic per total and work-group: they all fall on the same words (one per wavefront took
// 47 us on a batch of 40 scenes with 380,000 buckets, one per work-group takes 8).
constexpr int kStartsBlock = 1024;
__global__ __launch_bounds__(kStartsBlock) void bucket_starts(Buckets a) {
    __shared__ int part[kStartsBlock / 64][4], base[4];
    const int bk = blockIdx.x * kStartsBlock + threadIdx.x, w = threadIdx.x >> 6;
    const int k = bk < 2 * a.V ? a.cnt[bk] : 0;
    const bool column = k > 0 && (bk & 1) == 0;
    const int want[4] = {k > 0 ? 1 : 0, column ? k : 0, column ? 0 : k, column ? k + a.scol[(bk >> 1) + 1] - a.scol[bk >> 1] : 0};
    int at[4], sum;
    for (int c = 0; c < 4; ++c) {
        at[c] = wave_prefix(want[c], sum);
        if ((threadIdx.x & 63) == 0) part[w][c] = sum;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        sum = 0;
        for (int i = 0; i < kStartsBlock / 64; ++i) {
            const int x = part[i][threadIdx.x];
            part[i][threadIdx.x] = sum;
            sum += x;
        }
        base[threadIdx.x] = sum ? atomicAdd(a.totals + threadIdx.x, sum) : 0;
    }
    __syncthreads();
    if (k == 0) return;
    for (int c = 0; c < 4; ++c) at[c] += base[c] + part[w][c];
    a.list[at[0]] = bk;
    a.start[bk] = column ? at[1] : at[2];
    if (column) a.mstart[bk >> 1] = at[3];
}
__global__ void bucket_scatter(Buckets a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.nb) {
        const unsigned long long k = a.bkey[i];
        if (k != kNoKey)
            a.entries[a.start[2 * (int)(k >> a.kb)] + a.slot[i]] = ((k & ((1ull << a.kb) - 1)) << 32) | (unsigned)i;
    }
    if (i < a.ng) {
        const int v = a.gkey[i];
        if (v < a.V) a.entries[(size_t)a.nb + a.start[2 * v + 1] + a.slot[a.nb + i]] = (unsigned)i;
    }
}
// One work-group of two wavefronts per listed bucket (vertices in contact have 20 to 300 block
// records).  Every entry is placed by its rank, the number of smaller ones (all are distinct;
// a bitonic network by one wavefront took longer than everything else here): kBucketLds entries
// in LDS at a time, the result in LDS if they all fit.  Then kSumBlock entries at a time: their
// values into LDS, all loads in flight at once and neighbouring lanes reading neighbouring
// values, and a column's runs of equal rows, a lane per entry of the 3x3 block, zero entries
// skipped, with the flags of entries that received a nonzero value; a vertex's gradient by a lane
// per component.  Bound by the latency of one bucket's chain while the buckets are few.
// From the records to the sums: 5 + 5 + 63 us on four 20^3 cubes in contact and 25 us on two
// 11^3, where two scans, a sort by one wavefront, a thread per run and a thread per gradient
// took 223 and 82.
constexpr int kSumBlock = 128, kBucketLds = 512;
struct BucketLds {
    union {
        unsigned long long e[kBucketLds];
        double val[kSumBlock * 9];
    };
    unsigned long long sorted[kBucketLds];
    int start[kSumBlock + 1], heads[kSumBlock / 64];
};
// sorted[rank] of the bucket's entries [i0, i0 + N kSumBlock)
template <int N>
__device__ inline void place_entries(const unsigned long long* __restrict__ entries, int i0, int k, BucketLds& sh,
                                     unsigned long long* sorted) {
    const int t = threadIdx.x;
    unsigned long long v[N];
    int rank[N];
    for (int c = 0; c < N; ++c) {
        const int i = i0 + kSumBlock * c + t;
        v[c] = i < k ? entries[i] : 0ull;
        rank[c] = 0;
    }
    for (int j0 = 0; j0 < k; j0 += kBucketLds) {
        const int m = min(kBucketLds, k - j0);
        __syncthreads();
        for (int j = t; j < m; j += kSumBlock) sh.e[j] = entries[j0 + j];
        __syncthreads();
#pragma unroll 4
        for (int j = 0; j < m; ++j) {
            const unsigned long long x = sh.e[j];
#pragma unroll
            for (int c = 0; c < N; ++c) rank[c] += x < v[c] ? 1 : 0;
        }
    }
    for (int c = 0; c < N; ++c)
        if (i0 + kSumBlock * c + t < k) sorted[rank[c]] = v[c];
}
__device__ inline void place_bucket(const unsigned long long* __restrict__ entries, int k, BucketLds& sh, unsigned long long* sorted) {
    for (int i0 = 0; i0 < k; i0 += 4 * kSumBlock) {
        if (k - i0 <= kSumBlock) place_entries<1>(entries, i0, k, sh, sorted);
        else if (k - i0 <= 2 * kSumBlock) place_entries<2>(entries, i0, k, sh, sorted);
        else place_entries<4>(entries, i0, k, sh, sorted);
    }
    __syncthreads();
}
__device__ inline void sum_gradients(const Buckets& a, int v, int k, const unsigned long long* e, BucketLds& sh) {
    const int t = threadIdx.x;
    double* g = a.grad + 3 * (size_t)v + t;
    double sum = t < 3 ? *g : 0.0;
    for (int i0 = 0; i0 < k; i0 += kSumBlock) {
        const int m = min(kSumBlock, k - i0);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int q = t + kSumBlock * c;
            if (q < 3 * m) sh.val[q] = a.gval[(size_t)3 * (unsigned)e[i0 + q / 3] + q % 3];
        }
        __syncthreads();
        if (t < 3)
#pragma unroll 8
            for (int j = 0; j < m; ++j) sum += sh.val[3 * j + t];
        __syncthreads();
    }
    if (t < 3) *g = sum;
}
// The sums of a column's runs at s0, and how many there are.
__device__ inline int sum_column(const Buckets& a, int s0, int k, const unsigned long long* e, BucketLds& sh) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, l = lane / 9, c = lane - 9 * l;
    int u = 0;
    for (int i0 = 0; i0 < k; i0 += kSumBlock) {
        const int m = min(kSumBlock, k - i0), i = i0 + t;
#pragma unroll
        for (int x = 0; x < 9; ++x) {
            const int q = t + kSumBlock * x;
            if (q < 9 * m) sh.val[q] = a.cval[(size_t)9 * (unsigned)e[i0 + q / 9] + q % 9];
        }
        const bool head = i < k && (i == 0 || (e[i] >> 32) != (e[i - 1] >> 32));
        const unsigned long long heads = __ballot(head);
        if (lane == 0) sh.heads[w] = __popcll(heads);
        const int cont = i0 > 0 && (e[i0] >> 32) == (e[i0 - 1] >> 32) ? 1 : 0;    // the last chunk's last run goes on
        __syncthreads();
        const int nr = sh.heads[0] + sh.heads[1] + cont, r0 = s0 + u - cont;
        const int o = cont + (w ? sh.heads[0] : 0) + __popcll(heads & ((1ull << lane) - 1));
        if (head) {
            sh.start[o] = t;
            a.urow[r0 + o] = (int)(e[i] >> 32);
        }
        if (t == 0) {
            if (cont) sh.start[0] = 0;
            sh.start[nr] = m;
        }
        __syncthreads();
        for (int q = 7 * w; q < nr; q += 14) {
            const int r = q + l;
            const bool on = l < 7 && r < nr;
            double sum = 0.0;
            bool any = false;
            if (on) {
                if (r == 0 && cont) {
                    sum = a.uval[(size_t)9 * r0 + c];
                    any = (a.uflag[r0] >> c) & 1;
                }
                const int end = sh.start[r + 1];
                for (int j = sh.start[r]; j < end; ++j) {
                    const double x = sh.val[9 * j + c];
                    const bool nz = x != 0.0;
                    sum += nz ? x : 0.0;   // exact: an accumulator starting at +0 never holds -0
                    any |= nz;
                }
                a.uval[(size_t)9 * (r0 + r) + c] = sum;
            }
            const unsigned long long f = __ballot(on && any);
            if (on && c == 0) a.uflag[r0 + r] = (unsigned short)((f >> (9 * l)) & 0x1ffu);
        }
        u += nr - cont;
        __syncthreads();   // the LDS is the next chunk's, whose first run may read the last sum
    }
    return u;
}
__global__ __launch_bounds__(kSumBlock) void bucket_sums(Buckets a) {
    __shared__ BucketLds sh;
    const int n = a.totals[0];
    for (int t = blockIdx.x; t < n; t += gridDim.x) {
        const int bk = a.list[t], k = a.cnt[bk], s0 = a.start[bk];
        const size_t at = (size_t)(bk & 1 ? a.nb : 0) + s0;
        unsigned long long* sorted = k <= kBucketLds ? sh.sorted : a.sorted + at;
        int u = 0;   // a gradient bucket's count is cleared for the next assembly
        place_bucket(a.entries + at, k, sh, sorted);
        if (bk & 1) sum_gradients(a, bk >> 1, k, sorted, sh);
        else u = sum_column(a, s0, k, sorted, sh);
        if (threadIdx.x == 0) a.cnt[bk] = u;
        __syncthreads();   // the LDS is the next bucket's
    }
}

// Room for nb block and ng gradient records, and their buckets' counts cleared where the last
// assembly is not known to have left them so (a new buffer, a larger scene, an enqueue cut
// short).  Before the launches that write the records.
void bucket_records_prepare(Context& c, size_t nb, size_t ng) {
    const size_t ncnt = 2 * (size_t)c.sc.V + 4;   // counts, then the totals
    c.bucket_cnt.resize(ncnt);
    c.bucket_slot.resize(nb + ng + 1);
    if (c.bucket_cnt_clear < ncnt || c.bucket_cnt_ptr != c.bucket_cnt.p) {
        hipLaunchKernelGGL(zero_ints, dim3(blocks_for(ncnt, 256)), dim3(256), 0, c.stream, c.bucket_cnt.p, (int)ncnt);
        CIPC_CHECK_LAUNCH();
    }
    c.bucket_cnt_clear = 0;
    c.bucket_cnt_ptr = c.bucket_cnt.p;
}
// The nonzero and collision counts (c.coll) to pinned memory, for the host's next
// synchronisation.
void publish_nnz(Context& c, hipStream_t st) {
    c.pin_nnz.reserve(2);
    CIPC_HIP(hipMemcpyAsync(c.pin_nnz.p, c.coll.p, 2 * sizeof(int), hipMemcpyDeviceToHost, st));
    c.nnz_pending = true;
}
// The collision count of the assembly's set (c.coll[1]), on stream st.
void collision_count_launch(Context& c, hipStream_t st) {
    if (c.coll.n < 4) {
        c.coll.resize(4);
        hipLaunchKernelGGL(zero_ints, dim3(1), dim3(64), 0, st, c.coll.p + 2, 2);   // from then on each count leaves its sums cleared
    }
    hipLaunchKernelGGL(collision_count, dim3(kCountGroups), dim3(256), 0, st, c.dcnt.p + kDcSelf, c.self_set.p, c.coll.p);
    CIPC_CHECK_LAUNCH();
}

void finalize_csr(Context& c, bool count_collisions) {
    Scene& s = c.sc;
    const int V = s.V;
    const int nb = (int)c.ckey.n, ng = (int)c.gkey.n;
    if (count_collisions) collision_count_launch(c, c.stream);   // (else the caller has, on a stream of its own)
    // the contact records' sums: unique blocks per column, gradients into c.grad
    Buckets k;
    k.V = V; k.kb = s.kb; k.nb = nb; k.ng = ng; k.bkey = c.ckey.p; k.gkey = c.gkey.p;
    c.bucket_start.resize(3 * (size_t)V); c.bucket_list.resize(2 * (size_t)V);
    c.bucket_entries.resize((size_t)nb + ng + 1); c.bucket_sorted.resize((size_t)nb + ng + 1);
    c.urow.resize((size_t)nb + 1); c.uval.resize((size_t)9 * (nb + 1)); c.uflag.resize((size_t)nb + 1);
    k.cnt = c.bucket_cnt.p; k.totals = k.cnt + 2 * V; k.start = c.bucket_start.p; k.list = c.bucket_list.p; k.slot = c.bucket_slot.p;
    k.mstart = k.start + 2 * V; k.scol = c.sp.col_ptr.p;
    k.entries = c.bucket_entries.p; k.sorted = c.bucket_sorted.p; k.cval = c.cval.p; k.gval = c.gval.p;
    k.urow = c.urow.p; k.uval = c.uval.p; k.uflag = c.uflag.p; k.grad = c.grad.p;
    const int nmax = std::max(nb, ng);
    if (nmax > 0) {
        hipLaunchKernelGGL(bucket_starts, dim3(blocks_for(2 * (size_t)V, kStartsBlock)), dim3(kStartsBlock), 0, c.stream, k);
        hipLaunchKernelGGL(bucket_scatter, dim3(blocks_for(nmax, 256)), dim3(256), 0, c.stream, k);
        // no more work-groups than fit the chip at once
        const int groups = (int)std::min<size_t>(std::min<size_t>(2 * (size_t)V, (size_t)nb + ng), 256 * 10);
        hipLaunchKernelGGL(bucket_sums, dim3(groups), dim3(kSumBlock), 0, c.stream, k);
        CIPC_CHECK_LAUNCH();
    }
    // merged blocks and scalar entries, sized by their bounds (static blocks + contact records,
    // 9 entries each)
    const size_t mcap = (size_t)c.sp.nblocks + (size_t)nb + 1, nscan = 4 * (size_t)V + 2;
    c.merge_src.resize(mcap); c.merge_cnt.resize(nscan); c.mptr.resize(nscan);
    c.mrow.resize(mcap); c.mcol.resize(mcap); c.mval.resize(9 * mcap);
    c.outer.resize((size_t)3 * V + 1); c.inner.resize(9 * mcap); c.val.resize(9 * mcap); c.rhs.resize((size_t)3 * V);
    Merge a;
    a.V = V; a.nblocks = (int)c.sp.nblocks; a.nb = nb; a.scol = c.sp.col_ptr.p; a.srow = c.sp.row.p; a.sbv = c.sbv.p; a.sbf = c.sbf.p;
    a.ucnt = k.cnt; a.ustart = k.start; a.mstart = k.mstart; a.urow = k.urow; a.uval = k.uval; a.uflag = k.uflag; a.src = c.merge_src.p;
    a.count = c.merge_cnt.p; a.off = c.mptr.p; a.totals = k.totals; a.bt = s.bt.p; a.grad = c.grad.p;
    a.mrow = c.mrow.p; a.mcol = c.mcol.p; a.mval = c.mval.p; a.outer = c.outer.p; a.inner = c.inner.p; a.nnz_out = c.coll.p;
    a.val = c.val.p; a.rhs = c.rhs.p;
    hipLaunchKernelGGL(merge_count, dim3(blocks_for(V, 256)), dim3(256), 0, c.stream, a);
    CIPC_CHECK_LAUNCH();
    exclusive_scan_int(c, a.count, a.off, (int)nscan);   // mptr: the first V + 1
    hipLaunchKernelGGL(csr_fill, dim3(blocks_for((size_t)V * kFillLanes, 256)), dim3(256), 0, c.stream, a);
    CIPC_CHECK_LAUNCH();
    c.bucket_cnt_clear = c.bucket_cnt.n;
    // the counts are read with the caller's next synchronisation (or the caller publishes them)
    if (count_collisions) publish_nnz(c, c.stream);
}

}  // namespace cipc
