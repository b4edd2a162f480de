// solve.hip -- supernodal forward / diagonal / backward solve on the device-resident factors
// (aptp_solve, sparse/src/symmetric/solve.rs:57-326), for nrhs right-hand sides.
//
// The factors are read from each front's kept columns (the front itself for a root, else the
// copy of its first ne columns made at its level's end, same layout): L11 = F[0:ne, 0:ne] (unit
// lower, 2x2 off-diagonals zeroed), L21 = F[ne:m, 0:ne], row/column indices from the solve index.
//
// Each sweep is ONE launch over the whole assembly tree, run as a dataflow: work items are
// ordered so that every item depends only on items before it, each workgroup takes the next
// item with a ticket (atomic counter) when it starts, and waits for what it needs on flags and
// counters in device memory.  A waiting workgroup therefore only waits for workgroups that
// already run, so every wait ends (bounded in any case: a wait that exceeds its limit sets an
// error word the host reports instead of hanging).
//
//  forward (L y = b, solve.rs:89-92), per front with ne > 0:
//    diagonal item c  -- pulls the descendants' updates into the rows of column block c (the
//                        L21*x vectors Y of the fronts below, in postorder, as the reference
//                        subtracts them), streams L[c block rows, 0 : 128c] against the blocks
//                        already solved, solves the 128 x 128 unit triangle and publishes x_c;
//    rows item g      -- Y = L21[128 rows] * x, streamed block by block as they are published.
//  backward (D z = y, L^T x = z, solve.rs:97-141), per front:
//    column chunk item (C, h) -- partial products L21[256 rows of chunk h, block C]^T x_rows
//                        once every ancestor has finished;
//    diagonal item C  -- z = D^-1 y for its columns (MixedDiagonal::solve_in_place,
//                        diagonal.rs:312-365), minus the chunk partials in order, minus
//                        L[block C', block C]^T x_C' for the later blocks C' as they are
//                        published, then the 128 x 128 transposed unit triangle.
// A right-hand-side group of up to 8 columns shares every load of L.  All sums run in a fixed
// order: results do not depend on scheduling, nor on the number of columns.
//
// A single right-hand side is bound by the chain of diagonal blocks (97 of them on the way to the
// root of a Helmholtz 64^3 factor): a block's x is on its way to the next workgroup for about 2 us,
// its products take half a microsecond and its triangles one.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>

#include "../../include/rivrs_ldlt.h"
#include "rv_numeric.h"
#include "rv_poll.h"

namespace rv {

namespace {

constexpr int SB = 128;  // diagonal block of the blocked triangular solves (two 64-column halves)
constexpr int GH = 256;  // L21 rows per backward column-chunk item
constexpr int SPIN_LIMIT = 1 << 22;

// Item kinds.  A front with one diagonal block and at most FUSE_R rows of L21 is one fused item
// per sweep; larger fronts split into diagonal, rows and chunk items.
enum { IT_FDIAG = 0, IT_FROWS = 1, IT_FSMALL = 2, IT_BCHUNK = 3, IT_BDIAG = 4, IT_BSMALL = 5 };
constexpr int FUSE_R = 512;

// Everything the items of one front need, in one record (one dependent load after the item).
struct SolveFront {
    const double *F;     // front, lda = m
    const int *sidx;     // global index of local row i
    const int8_t *dkind;
    const double *ddiag, *doff;
    long long wbase;     // offset of the front's columns in W / Xb
    long long ybase;     // offset of the front's L21 rows in Y
    long long pbase;     // offset of the front's chunk partials in P
    int m, ne;
    int fbase;           // first block flag of the front
    int nchk;            // backward: chunks per column block
    int ech0, ech1;      // effective children (nearest descendants with ne > 0) in ech
    int epar;            // effective parent or -1
    int epar_nblk;       // its done target in the backward sweep (on top of the forward's)
};

// The solve plan as the kernels see it.
struct PlanDev {
    const SolveFront *sf;
    const int2 *ech;             // (child front, its forward done target)
    const int *ptr;              // pull lists: Y entries per global index
    const long long *ent;
    int nfront, nflag;
};

// Counters, zeroed by k_solve_start; every array holds one slice per RHS group.
struct SyncDev {
    int *tick;   // [2] ticket counters of the two sweeps
    int *err;    // [1] set when a wait exceeded its limit
    int *done;   // forward: rows items of the front finished; backward, counting on: its blocks
    int *bgc;    // backward: chunk items of the block finished
};

// Data that one workgroup of a sweep writes and another reads within the same launch (x blocks,
// Y, chunk partials) goes through device-coherent accesses: stores and loads with device scope
// (they bypass the per-XCD L2, whose copies another XCD's writes would leave stale), so no cache
// maintenance fence is needed.  The blocks of x along the chain are polled themselves (UNSET,
// below).  For the rest a producer stores its data, waits until its stores have completed
// (s_waitcnt), joins a workgroup barrier, and one thread bumps a counter with a device-scope
// atomic; a consumer's thread spins on the counter with device-scope loads, and after a workgroup
// barrier every thread reads the data with device-scope loads.  The factor L is never written
// during a solve and is read through the caches as usual.
__device__ __forceinline__ double ld_co(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void st_co(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// every thread's device-coherent stores complete, then the workgroup barrier
__device__ __forceinline__ void stores_done_barrier() {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// A thread waits until *p >= target; the caller follows with a workgroup barrier.
__device__ __forceinline__ void wait_at_least(const int *p, int target, int *err) {
    long long it = 0;
    while (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
        if ((++it & 63) == 0 &&
            (it > SPIN_LIMIT || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
            atomicOr(err, 1);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

// after stores_done_barrier(), by one thread
__device__ __forceinline__ void publish_add(int *p) {
    __hip_atomic_fetch_add(p, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Blocks of x pass between workgroups without a flag: W and Xb start a solve filled with UNSET,
// a signalling NaN that no arithmetic returns, and a reader polls the words it needs until none
// is UNSET.  A flag costs the writer the wait for its stores and the reader a second trip.
constexpr unsigned long long UNSET = 0x7FF4A5A55A5A5A4Aull;
__device__ __forceinline__ unsigned long long ld_bits(const double *p) {
    return __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish_value(double *p, double v) {
    unsigned long long b = (unsigned long long)__double_as_longlong(v);
    if (b == UNSET) b = 0x7FF8000000000000ull;  // (an input's own NaN)
    __hip_atomic_store((unsigned long long *)p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int take_ticket(int *tick) {
    __shared__ int s_t;
    if (threadIdx.x == 0) s_t = atomicAdd(tick, 1);
    __syncthreads();
    return s_t;
}

// A solve's vectors hold group g of right-hand sides (nq columns from q0 = g wq on) in nq
// consecutive entries per index, group after group: column q of index i is at
// q0 total + i nq + (q - q0), and a gather of an index serves the whole group.

// Start of a solve: x_perm[i] = rhs[perm_fwd[i]] (* s[i]) (solver.rs:396-410) for every RHS
// column, the sweeps' counters cleared, and the published vectors (W and Xb, nfill entries from
// fill on) set to UNSET.
__global__ void k_solve_start(const double *__restrict__ rhs, long long ld, double *__restrict__ xp, long long n,
                              int nrhs, int wq, const int *__restrict__ pf, const double *__restrict__ s,
                              int *__restrict__ sync, long long nsync, unsigned long long *__restrict__ fill,
                              long long nfill) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int q0 = blockIdx.y * wq, nq = min(wq, nrhs - q0);
    const long long step = (long long)gridDim.x * blockDim.x;
    if (blockIdx.y == 0)
        for (long long e = i; e < nsync; e += step) sync[e] = 0;
    for (long long e = blockIdx.y * step + i; e < nfill; e += step * gridDim.y) fill[e] = UNSET;
    if (i >= n) return;
    const int p = pf[i];
    const double si = s ? s[i] : 1.0;
#pragma unroll 4
    for (int q = 0; q < nq; ++q) {
        double v = rhs[p + (q0 + q) * ld];
        if (s) v *= si;
        xp[q0 * n + i * nq + q] = v;
    }
}

// rhs[perm_fwd[i]] = x_perm[i] (* s[i])  (solver.rs:416-425)
__global__ void k_perm_out(double *__restrict__ rhs, long long ld, const double *__restrict__ xp, long long n,
                           int nrhs, int wq, const int *__restrict__ pf, const double *__restrict__ s) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int q0 = blockIdx.y * wq, nq = min(wq, nrhs - q0);
    if (i >= n) return;
    const int p = pf[i];
    const double si = s ? s[i] : 1.0;
#pragma unroll 4
    for (int q = 0; q < nq; ++q) {
        double v = xp[q0 * n + i * nq + q];
        if (s) v *= si;
        rhs[p + (q0 + q) * ld] = v;
    }
}

// Pull of columns that no front eliminated (unresolved delays at the roots).
__global__ void k_pull_rows(const int *__restrict__ rows, int nrows, const int *__restrict__ ptr,
                            const long long *__restrict__ ent, const double *__restrict__ Y,
                            long long ytotal, double *__restrict__ x, long long n, int nrhs, int wq) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int q0 = blockIdx.y / wq * wq, nq = min(wq, nrhs - q0), q = blockIdx.y - q0;
    if (i >= nrows) return;
    const int t = rows[i];
    double v = x[q0 * n + (long long)t * nq + q];
    for (int e = ptr[t]; e < ptr[t + 1]; ++e) v -= Y[q0 * ytotal + ent[e] * nq + q];
    x[q0 * n + (long long)t * nq + q] = v;
}

// Inverses of the diagonal triangles.  Every 64 x 64 unit lower triangle T of L11 the solve
// uses (columns jb .. jb + n - 1 of a front, n <= 64) is inverted once per factorization, at the
// first solve after it, and X = T^-1 (unit lower) is kept in the unused upper triangle of the
// same diagonal block: X(i, j), i > j, at front position (jb + j, jb + i).  The sweeps then form
// x = X w and x = X^T w as dot products, where the substitution needed 63 dependent steps.
// (Every other reader of a front -- factorization kernels, extend-add, exports -- uses its lower
// triangle only.)
// One wavefront per triangle: lane c holds column c of X in registers and forms it column by
// column of T (x = e_c; for j = 0, 1, ...: x_i -= T(i, j) x_j for i > j, as one FMA per entry),
// with T in LDS by columns (Tt[j][i] = T(i, j)), read by all lanes at the same address.  The
// triangle's order n is rounded up to S = 16, 32 or 64 (rows and columns from n on are zeros and
// are not stored back), so the loops are fixed and unrolled.  The updates run in groups of eight
// rows of one column, each group's T entries loaded three groups ahead; a scheduling barrier after
// every group keeps the unrolled loop's 2016 loads from being hoisted all at once.  Global loads
// and stores go through a buffer resource based at the triangle, with an out-of-range offset for
// the entries a lane skips: no divergent branch, which would keep x's registers apart per branch.
template <int S, int J, int I0>
struct InvNext {
    static constexpr bool more = I0 + 8 < S;
    static constexpr int j = more ? J : J + 1;
    static constexpr int i0 = more ? I0 + 8 : J + 2;
    static constexpr bool valid = j < S - 1;
};
template <int S, int J, int I0>
__device__ __forceinline__ void inv_load(double (&c)[8], const double (*Tt)[64]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = (I0 + u < S) ? Tt[J][I0 + u < S ? I0 + u : 0] : 0.0;
}
template <int S, int J, int I0>
__device__ __forceinline__ void inv_groups(double (&x)[S], const double (*Tt)[64], const double (&c0)[8],
                                           const double (&c1)[8], const double (&c2)[8]) {
    using N1 = InvNext<S, J, I0>;
    using N2 = InvNext<S, N1::j, N1::i0>;
    using N3 = InvNext<S, N2::j, N2::i0>;
    double c3[8] = {};
    if constexpr (N1::valid && N2::valid && N3::valid) inv_load<S, N3::j, N3::i0>(c3, Tt);
    const double xj = x[J];
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (I0 + u < S) x[I0 + u] = fma(-c0[u], xj, x[I0 + u]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (N1::valid) inv_groups<S, N1::j, N1::i0>(x, Tt, c1, c2, c3);
}

template <int S>
__device__ __forceinline__ void invert_unit_lower(double (*Tt)[64], __amdgpu_buffer_rsrc_t rb, size_t lda, int n) {
    const int l = threadIdx.x;
    constexpr int OUT = 0x7FFFFFF8;  // beyond the resource: the load returns 0, the store is dropped
    // lane l: row l of T, columns j < min(l, S - 1), 16 loads in flight per round trip (n <= S)
#pragma unroll
    for (int j0 = 0; j0 < S - 1; j0 += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int j = j0 + u;
            const int off = (l < n && j < l) ? (int)((l + (size_t)j * lda) * sizeof(double)) : OUT;
            v[u] = (j < S - 1) ? __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rb, off, 0, 0)) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (j0 + u < S - 1) Tt[j0 + u][l] = v[u];
    }
    __syncthreads();
    double x[S];
#pragma unroll
    for (int i = 0; i < S; ++i) x[i] = (i == l) ? 1.0 : 0.0;
    using N1 = InvNext<S, 0, 1>;
    using N2 = InvNext<S, N1::j, N1::i0>;
    double c0[8], c1[8], c2[8];
    inv_load<S, 0, 1>(c0, Tt);
    inv_load<S, N1::j, N1::i0>(c1, Tt);
    inv_load<S, N2::j, N2::i0>(c2, Tt);
    inv_groups<S, 0, 1>(x, Tt, c0, c1, c2);
    // X(i, l), i > l, at front position (jb + l, jb + i)
#pragma unroll
    for (int i = 1; i < S; ++i) {
        const int off = (i > l && i < n) ? (int)((l + (size_t)i * lda) * sizeof(double)) : OUT;
        typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x[i]), rb, off, 0, 0);
    }
}

// One launch per order class S (the host groups the triangles), so each holds only its LDS.
template <int S>
__global__ __launch_bounds__(64) void k_diag_inverse(const SolveFront *__restrict__ sf,
                                                     const int4 *__restrict__ tris) {
    __shared__ __align__(16) double Tt[S - 1][64];
    const int4 t = tris[blockIdx.x];
    const SolveFront &Fr = sf[t.x];
    const int jb = t.y, n = t.z;
    const size_t lda = (size_t)Fr.m;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double *>(Fr.F) + jb + (size_t)jb * lda, (short)0, 0x7FFFFFF0, 0x00020000);
    invert_unit_lower<S>(Tt, rb, lda, n);
}

// ---------------------------------------------------------------------------
// Products on the matrix cores.  A workgroup serves W = 4 or 8 right-hand sides (nq <= W of them in
// use); a wavefront owns 16-row tiles of the result.  The four blocks of v_mfma_f64_4x4x4 take 16
// rows of L as one fragment -- lane l holds L(row l & 15, k = l >> 4) -- and four columns of x,
// the same for all blocks; its four products are four FMAs in the order k = 0, 1, 2, 3, so a
// column's result does not depend on W or on its neighbours.  One fragment of L serves all W
// columns; on the VALU every product took an LDS read of x.
// Why not v_mfma_f64_16x16x4 and 16 columns: a sweep is bound by its chain of diagonal blocks, and a
// step of the chain takes as long as the products of one workgroup.  Helmholtz 40^3, both sweeps:
// 8 right-hand sides 2.58 ms on the VALU, 1.37 on the wide instruction, 0.66 in groups of 4 (one
// column 0.87 on the VALU, 0.58 now; 64 columns 5.39 and 1.63).
// Element e of lane l is row tile_row(l) of the tile, column tile_col(l) + e: a lane's columns are
// adjacent and come with one read.
// ---------------------------------------------------------------------------
template <int W>
struct Tile {
    double e[W / 4];
};
template <int W>
__device__ __forceinline__ Tile<W> tile_zero() {
    Tile<W> t;
#pragma unroll
    for (int e = 0; e < W / 4; ++e) t.e[e] = 0.0;
    return t;
}
template <int W>
__device__ __forceinline__ int tile_col(int lane) { return W / 4 * (lane & 3); }
__device__ __forceinline__ int tile_row(int lane) { return 4 * ((lane >> 2) & 3) + (lane >> 4); }
template <int W>
__device__ __forceinline__ Tile<W> operator+(const Tile<W> &a, const Tile<W> &b) {
    Tile<W> t;
#pragma unroll
    for (int e = 0; e < W / 4; ++e) t.e[e] = a.e[e] + b.e[e];
    return t;
}
template <int W>
__device__ __forceinline__ Tile<W> operator-(const Tile<W> &a, const Tile<W> &b) {
    Tile<W> t;
#pragma unroll
    for (int e = 0; e < W / 4; ++e) t.e[e] = a.e[e] - b.e[e];
    return t;
}
// x: the lane's first entry of the fragment's row
template <int W>
__device__ __forceinline__ void mma(double a, const double *x, Tile<W> &c) {
#pragma unroll
    for (int e = 0; e < W / 4; ++e) c.e[e] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, x[e], c.e[e], 0, 0, 0);
}
// a tile to and from W-wide rows
template <int W>
__device__ __forceinline__ void tile_store(double *rows, const Tile<W> &t) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int e = 0; e < W / 4; ++e) rows[tile_row(lane) * W + tile_col<W>(lane) + e] = t.e[e];
}
template <int W>
__device__ __forceinline__ Tile<W> tile_load(const double *rows) {
    const int lane = threadIdx.x & 63;
    Tile<W> t;
#pragma unroll
    for (int e = 0; e < W / 4; ++e) t.e[e] = rows[tile_row(lane) * W + tile_col<W>(lane) + e];
    return t;
}

// Loads of L go through buffer resources based at a block of columns and ending after its last
// valid column: columns past the end and masked lanes (offset OUT) read zero, without a branch.
constexpr unsigned OUT = 0x7FFFFFF8u;  // (column offsets added to it stay past every range)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t cols_rsrc(const gdouble *L, size_t lda, size_t c0, int ncols) {
    const size_t bytes = (size_t)ncols * lda * sizeof(double);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>((const double *)(L + c0 * lda)), (short)0,
                                             (int)(bytes < 0x7FFFFFF0 ? bytes : 0x7FFFFFF0), 0x00020000);
}
__device__ __forceinline__ double buf_ld(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

// Row order of x for the transposed products (see TCols)
__device__ __forceinline__ int tcol_pos(int row) { return (row & ~7) | ((row & 1) << 2) | ((row >> 1) & 3); }

// A block's n rows of x (row stride nq) on their way to LDS.  ask loads the words without waiting
// for them (AHEAD: while the block before is used, so that a block published long ago costs a reader
// behind the chain no trip of its own); take polls until all are set and stores them to xb (row stride W, zeros for rows and columns that
// do not exist; TCOL: rows in the order of tcol_pos), ending with the barrier.  near: the block is
// one of the reader's last NEAR steps of the chain and is polled by every thread; otherwise a
// wavefront waits for one word of it first, a trip more.
constexpr int NEAR = 3;
template <int W, bool TCOL = false>
struct XBlock {
    static constexpr int NI = SB * W / 256;
    static constexpr bool AHEAD = W == 4;  // (wider, the registers are short)
    const double *src;
    int n, nq;
    unsigned long long v[NI];
    __device__ __forceinline__ void ask(const double *src_, int n_, int nq_) {
        src = src_, n = n_, nq = nq_;
        reload();
    }
    __device__ __forceinline__ void reload() {
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int e = tid + 256 * i, row = e / W, q = e % W;
            v[i] = (row < n && q < nq) ? ld_bits(src + (size_t)row * nq + q) : 0ull;
        }
    }
    __device__ __forceinline__ void take(bool near, double *xb, int *err) {
        const int tid = threadIdx.x;
        SpinBudget budget{SPIN_LIMIT};
        wait_words(
            near,
            [&] {
                bool bad = false;
#pragma unroll
                for (int i = 0; i < NI; ++i) bad |= v[i] == UNSET;
                return (bool)__any(bad);
            },
            [&] { return ld_bits(src + (size_t)n * nq - 1) == UNSET; }, [&] { reload(); },
            [&] {
                if (budget.spent([&] { return __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; })) {
                    atomicOr(err, 1);
                    return true;
                }
                __builtin_amdgcn_s_sleep(1);
                return false;
            });
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int e = tid + 256 * i;
            xb[TCOL ? tcol_pos(e / W) * W + e % W : e] = __longlong_as_double((long long)v[i]);
        }
        __syncthreads();
    }
};

// Rows of a front times a chunk of 32 columns: two sums of 16 products, added and subtracted from
// acc (columns ascending).  a[t][s]: fragment of tile t, columns 4s .. 4s + 3; xb: the chunk's x.
template <int W>
__device__ __forceinline__ void fwd_chunk(const double (&a)[2][8], const double *xb, Tile<W> (&acc)[2]) {
    const int lane = threadIdx.x & 63, b0 = (lane >> 4) * W + tile_col<W>(lane);
    Tile<W> p[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) p[t][0] = p[t][1] = tile_zero<W>();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const double *x0 = xb + 4 * s * W + b0, *x1 = x0 + 16 * W;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            mma<W>(a[t][s], x0, p[t][0]);
            mma<W>(a[t][4 + s], x1, p[t][1]);
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t] = acc[t] - (p[t][0] + p[t][1]);
}

// acc -= L[r0 : r0 + nr, 0 : ncols] x, wavefront w forming rows 32w .. 32w + 31.  WAIT: x comes
// block by block from src as it is published; else (ncols <= SB) the caller has filled xs.  A whole
// block of L is in flight ahead of the products: when a block's x arrives, which ends a step of the
// chain, only products remain.  (With one chunk in flight a workgroup took 6 us a block and fell
// behind the chain, whose step is 3 to 5 us.)
template <int W, bool WAIT>
__device__ __forceinline__ void fwd_rows(const gdouble *L, size_t lda, int r0, int nr, int ncols, const double *src,
                                         int nq, Tile<W> (&acc)[2], double *xs, int *err) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool act = 32 * wv < nr;  // (the wavefront has rows)
    const int nblk = (ncols + SB - 1) / SB;
    const unsigned col = 8u * (unsigned)lda;
    unsigned off[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int row = 32 * wv + 16 * t + (lane & 15);
        off[t] = row < nr ? 8u * (unsigned)(r0 + row) + (unsigned)(lane >> 4) * col : OUT;
    }
    auto load = [&](int blk, int ch, double (&v)[2][8]) {
        const __amdgpu_buffer_rsrc_t r = cols_rsrc(L, lda, (size_t)blk * SB, min(SB, ncols - blk * SB));
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < 8; ++s) v[t][s] = buf_ld(r, off[t] + (unsigned)(32 * ch + 4 * s) * col);
    };
    // chunk ch of the current block in a[ch]; once used, its registers take the next block's
    double a[4][2][8];
    if (act) {
#pragma unroll
        for (int ch = 0; ch < 4; ++ch)
            if (32 * ch < ncols) load(0, ch, a[ch]);
    }
    XBlock<W> X;
    if (WAIT && X.AHEAD) X.ask(src, min(SB, ncols), nq);
    for (int blk = 0; blk < nblk; ++blk) {
        const int n = min(SB, ncols - blk * SB), next = ncols - (blk + 1) * SB;
        double *xb = xs + (blk & 1) * (SB * W);
        if (WAIT && !X.AHEAD) X.ask(src + (size_t)blk * SB * nq, n, nq);
        if (WAIT) X.take(blk + NEAR >= nblk, xb, err);
        if (WAIT && X.AHEAD && next > 0) X.ask(src + (size_t)(blk + 1) * SB * nq, min(SB, next), nq);
        if (!act) continue;
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
            if (32 * ch < n) fwd_chunk<W>(a[ch], xb + 32 * ch * W, acc);
            if (32 * ch < next) load(blk + 1, ch, a[ch]);
        }
    }
}

// The diagonal block [jb, jb + nb): fragments of the inverses of its two unit triangles (kept by
// k_diag_inverse in the block's upper triangle) in LDS, each read only by the wavefront that
// stored it, and of the tile C = L[jb + 64 : jb + 128, jb : jb + 64] between them in registers.
// Wavefront w forms rows 16w .. 16w + 15 of both halves; a product with a triangle is four sums,
// over the columns 16r .. 16r + 15 (r = 0 .. 3), of which those on the other side of the diagonal
// are empty and not stored: 40 fragments a triangle.  C_EARLY: C is loaded with the triangles;
// otherwise, where its registers are needed until then, after the block's other products
// (load_c), and its lines only touched here.
constexpr int TFRAG = 40 * 64;
template <bool FWD, bool C_EARLY>
struct Diag {
    double c[16];
    double *tri;  // the wavefront's fragments of triangle A; B's TFRAG later
    int n1, n2;
    static __device__ __forceinline__ bool has(int r, int w) { return FWD ? r <= w : r >= w; }
    __device__ __forceinline__ void load(const gdouble *L, size_t lda, int jb, int nb, double *frags) {
        const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int i = 16 * w + (lane & 15), k = lane >> 4;
        n1 = min(64, nb), n2 = nb - n1;
        tri = frags + (FWD ? 2 * w * (w + 1) : 16 * w - 2 * w * (w - 1)) * 64 + lane;
        const __amdgpu_buffer_rsrc_t ra = cols_rsrc(L, lda, jb, nb);
        const unsigned col = 8u * (unsigned)lda;
        auto half = [&](int h, int n, double (&v)[16]) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (has(r, w)) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const int j = 16 * r + 4 * s + k;
                        const int x = FWD ? i : j, y = FWD ? j : i;  // inverse entry (x, y), kept at (y, x)
                        v[4 * r + s] = buf_ld(ra, y < x && x < n ? 8u * (unsigned)(jb + h + y) + (unsigned)(h + x) * col : OUT);
                    }
                }
        };
        double a[16], b[16], touch = 0.0;
        half(0, n1, a);
        if (n2 > 0) {
            half(64, n2, b);
            if (C_EARLY) load_c(L, lda, jb);
            else touch = buf_ld(ra, 16 * k < n2 ? 8u * (unsigned)(jb + 64 + 16 * k) + (unsigned)i * col : OUT);
        }
        double *t = tri;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (has(r, w)) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    t[0] = a[4 * r + s];
                    if (n2 > 0) t[TFRAG] = b[4 * r + s];
                    t += 64;
                }
            }
        if (!C_EARLY) asm volatile("" ::"v"(touch));
    }
    __device__ __forceinline__ void load_c(const gdouble *L, size_t lda, int jb) {
        const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int i = 16 * w + (lane & 15), k = lane >> 4;
        const __amdgpu_buffer_rsrc_t ra = cols_rsrc(L, lda, jb, min(SB, n1 + n2));
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const int x = FWD ? i : 4 * s + k, y = FWD ? 4 * s + k : i;  // C(x, y)
            c[s] = buf_ld(ra, x < n2 ? 8u * (unsigned)(jb + 64 + x) + 8u * (unsigned)y * (unsigned)lda : OUT);
        }
    }
    // sum_j X(i, j) w_j (j != i) of half h, w in LDS (row stride W)
    template <int W>
    __device__ __forceinline__ Tile<W> tri_sum(int h, const double *ws) const {
        const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const double *t = tri + h * TFRAG;
        const double *x = ws + (64 * h + (lane >> 4)) * W + tile_col<W>(lane);
        Tile<W> a[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            a[r] = tile_zero<W>();
            if (has(r, w)) {
#pragma unroll
                for (int s = 0; s < 4; ++s) mma<W>(t[64 * s], x + (16 * r + 4 * s) * W, a[r]);
                t += 256;
            }
        }
        return (a[0] + a[1]) + (a[2] + a[3]);
    }
};

// Sum of leaf(r0) .. leaf(r0 + N - 1) as a binary tree
template <int N, class T, class F>
__device__ __forceinline__ T tree_sum(int r0, F &&leaf) {
    if constexpr (N == 1) {
        return leaf(r0);
    } else {
        const T x = tree_sum<N / 2, T>(r0, leaf);
        const T y = tree_sum<N / 2, T>(r0 + N / 2, leaf);
        return x + y;
    }
}
template <int W>
struct Tile2 {
    Tile<W> t[2];
};
template <int W>
__device__ __forceinline__ Tile2<W> operator+(const Tile2<W> &a, const Tile2<W> &b) {
    return Tile2<W>{{a.t[0] + b.t[0], a.t[1] + b.t[1]}};
}

// Transposed products: rows r0 .. r0 + nr - 1 (nr <= 128, r0 > 0) times columns c0 .. c0 + ncols - 1
// (at most 128; wavefront w forms columns 32w .. 32w + 31), x of the rows in xs.  A 16-byte load
// takes 64 bytes of each of 16 columns: rows 8s + 2k and 8s + 2k + 1 in lane group k, so the four
// even and the four odd rows of eight are a fragment each, and xs holds its rows in that order
// (tcol_pos).  Every fragment's sum is a leaf; the 32 leaves are added as a binary tree.
template <int W>
struct TCols {
    unsigned off[2];
    int nr, row0;
    __amdgpu_buffer_rsrc_t rs;
    double a[4][8][2];  // leaves 8g .. 8g + 7 in a[g]
    __device__ __forceinline__ void at(const gdouble *L, size_t lda, int r0, int nr_, int c0, int ncols) {
        const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        rs = cols_rsrc(L, lda, c0, ncols);
        nr = nr_;
        row0 = 2 * (lane >> 4);
#pragma unroll
        for (int t = 0; t < 2; ++t)
            off[t] = 8u * (unsigned)(r0 + row0) + (unsigned)(32 * wv + 16 * t + (lane & 15)) * 8u * (unsigned)lda;
    }
    __device__ __forceinline__ void load(int g) {
        typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
        typedef double f64x2 __attribute__((ext_vector_type(2)));
        auto pair = [&](unsigned o) { return __builtin_bit_cast(f64x2, __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)o, 0, 0))); };
        if (32 * g + 32 <= nr) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f64x2 v = pair(off[t] + 8u * (unsigned)(32 * g + 8 * s));
                    a[g][2 * s][t] = v[0];
                    a[g][2 * s + 1][t] = v[1];
                }
        } else {
            // a last odd row comes as the second of the pair before it
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int row = 32 * g + 8 * s + row0;
                const bool in0 = row < nr, in1 = row + 1 < nr;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f64x2 v = pair(in0 ? off[t] + 8u * (unsigned)(32 * g + 8 * s) - (in1 ? 0u : 8u) : OUT);
                    a[g][2 * s][t] = in1 ? v[0] : v[1];
                    a[g][2 * s + 1][t] = in1 ? v[1] : 0.0;
                }
            }
        }
    }
    __device__ __forceinline__ void load_all() {
#pragma unroll
        for (int g = 0; g < 4; ++g)
            if (32 * g < nr) load(g);
    }
    __device__ __forceinline__ Tile<W> sum(int g, int t, const double *xs) const {
        const int lane = threadIdx.x & 63;
        const double *x = xs + (lane >> 4) * W + tile_col<W>(lane);
        return tree_sum<8, Tile<W>>(0, [&](int r) {
            Tile<W> p = tile_zero<W>();
            mma<W>(a[g][r][t], x + 4 * (8 * g + r) * W, p);
            return p;
        });
    }
    // the sum over the rows; with a next tile (rows nr1 > 0 from r1, same columns), each group's
    // registers take its leaves once they are used
    __device__ __forceinline__ Tile2<W> step(const double *xs, int dr, int nr1) {
        Tile2<W> s[4];
        const int n = nr;
#pragma unroll
        for (int t = 0; t < 2; ++t) off[t] += 8u * (unsigned)dr;
        nr = nr1;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                s[g].t[t] = tile_zero<W>();
                if (32 * g < n) s[g].t[t] = sum(g, t, xs);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (32 * g < nr1) load(g);
            if (g & 1) s[g - 1] = s[g - 1] + s[g];
        }
        return s[0] + s[2];
    }
};


// ===========================================================================
// Forward sweep (one launch): ticket order = item order.
// ===========================================================================
template <int W>
__global__ __launch_bounds__(256, 2) void k_fwd_sweep(PlanDev P, const int4 *__restrict__ items, int nwork, int ngrp,
                                                      int nrhs, int wq, const double *__restrict__ x, long long n,
                                                      double *__restrict__ Wx, long long wtotal,
                                                      double *__restrict__ Y, long long ytotal, SyncDev S) {
    constexpr int NE = W / 4, NP = 2 * NE, NU = 16 / NP;
    const int t = take_ticket(S.tick);
    if (t >= nwork) return;
    const int4 it = items[t / ngrp];
    const int grp = t % ngrp, q0 = grp * wq, nq = min(wq, nrhs - q0);
    const int li = it.x;
    const SolveFront &Fr = P.sf[li];
    const int ne = Fr.ne, m = Fr.m;
    const size_t lda = (size_t)m;
    const gdouble *L = gbl(Fr.F);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int trow = tile_row(lane), qc = tile_col<W>(lane);
    double *Wf = Wx + (size_t)q0 * wtotal + (size_t)Fr.wbase * nq;
    double *Yg = Y + (size_t)q0 * ytotal;
    __shared__ __align__(16) double xs[2 * SB * W];
    __shared__ double frags[2 * TFRAG];
    Tile<W> acc[2] = {tile_zero<W>(), tile_zero<W>()};
    auto store_rows = [&](const Tile<W> (&a)[2], int r0, int nr) {  // Y of 128 rows of L21
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                const int row = 32 * wv + 16 * tt + trow, q = qc + e;
                if (row < nr && q < nq) st_co(Yg + (size_t)(Fr.ybase + (r0 - ne) + row) * nq + q, -a[tt].e[e]);
            }
    };
    if (it.y == IT_FROWS) {  // 128 rows of L21
        const int r0 = ne + it.z * SB, nr = min(SB, m - r0);
        fwd_rows<W, true>(L, lda, r0, nr, ne, Wf, nq, acc, xs, S.err);
        store_rows(acc, r0, nr);
        stores_done_barrier();
        if (tid == 0) publish_add(S.done + (size_t)grp * P.nfront + li);
        return;
    }
    const int j0 = it.z * SB, nb = min(SB, ne - j0);
    // The lists to pull, and what does not depend on the children, ahead of the wait for them
    int e0[NP], e1[NP];
    long long ent[NP][NU];
    double xv[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int row = 32 * wv + 16 * (p / NE) + trow, q = qc + p % NE;
        e0[p] = e1[p] = 0;
        xv[p] = 0.0;
        if (row < nb && q < nq) {
            const int tg = gbl(Fr.sidx)[j0 + row];
            if ((unsigned)tg < (unsigned)n) {
                e0[p] = P.ptr[tg];
                e1[p] = P.ptr[tg + 1];
                xv[p] = x[(size_t)q0 * n + (size_t)tg * nq + q];
            } else {
                atomicOr(S.err, 2);  // an index outside the system: the solve plan does not fit the fronts
            }
        }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int u = 0; u < NU; ++u) ent[p][u] = e0[p] + u < e1[p] ? P.ent[e0[p] + u] : 0;
    Diag<true, W == 4> dg;
    dg.load(L, lda, j0, nb, frags);
    // the descendants' Y vectors are complete once the effective children are
    if (wv == 0) {
        for (int e = Fr.ech0 + lane; e < Fr.ech1; e += 64) {
            const int2 ch = P.ech[e];
            wait_at_least(S.done + (size_t)grp * P.nfront + ch.x, ch.y, S.err);
        }
    }
    __syncthreads();
    // pull of the descendants' updates: x[t] - sum of the Y entries of global index t = sidx[i], in
    // list order (postorder of the fronts that produced them), a lane's rows in step
    {
        double sum[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) sum[p] = 0.0;
        for (;;) {
            bool more = false;
            double y[NP][NU];
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int u = 0; u < NU; ++u) {
                    y[p][u] = e0[p] + u < e1[p] ? ld_co(Yg + (size_t)ent[p][u] * nq + qc + p % NE) : 0.0;
                    // the next round's
                    ent[p][u] = e0[p] + NU + u < e1[p] ? P.ent[e0[p] + NU + u] : 0;
                }
#pragma unroll
            for (int p = 0; p < NP; ++p) {
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    if (e0[p] + u < e1[p]) sum[p] += y[p][u];
                e0[p] += NU;
                more |= e0[p] < e1[p];
            }
            if (!__any(more)) break;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) acc[p / NE].e[p % NE] = xv[p] - sum[p];
    }
    if (it.y == IT_FDIAG && j0 > 0) fwd_rows<W, true>(L, lda, j0, nb, j0, Wf, nq, acc, xs, S.err);
    if (W != 4 && dg.n2 > 0) dg.load_c(L, lda, j0);
    // The block's w, then its x.  The half of xs that the last block of x did not use is free.
    const int lastb = max(j0 / SB - 1, 0);
    double *ws = xs + ((lastb + 1) & 1) * (SB * W), *xo = xs + (lastb & 1) * (SB * W);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) tile_store<W>(ws + (32 * wv + 16 * tt) * W, acc[tt]);
    __syncthreads();
    // later blocks and the rows items of this front read a published x; a fused front's x stays in
    // LDS for its own rows, and W is read by the next launch
    auto finish = [&](int h, int nn, const Tile<W> &v) {
        tile_store<W>(xo + (64 * h + 16 * wv) * W, v);
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int row = 16 * wv + trow, q = qc + e;
            if (row < nn && q < nq) {
                double *p = Wf + (size_t)(j0 + 64 * h + row) * nq + q;
                if (it.y == IT_FDIAG) publish_value(p, v.e[e]);
                else *p = v.e[e];
            }
        }
    };
    auto own = [&](int h) { return tile_load<W>(ws + (64 * h + 16 * wv) * W); };
    finish(0, dg.n1, own(0) + dg.template tri_sum<W>(0, ws));
    if (dg.n2 > 0) {
        __syncthreads();
        Tile<W> p[4];
        const double *xa = xo + (lane >> 4) * W + qc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = tile_zero<W>();
#pragma unroll
            for (int s = 0; s < 4; ++s) mma<W>(dg.c[4 * r + s], xa + (16 * r + 4 * s) * W, p[r]);
        }
        const Tile<W> wb = own(1) - (((p[0] + p[1]) + p[2]) + p[3]);
        tile_store<W>(ws + (64 + 16 * wv) * W, wb);
        __syncthreads();
        finish(1, dg.n2, wb + dg.template tri_sum<W>(1, ws));
    } else if (it.y == IT_FSMALL) {
        tile_store<W>(xo + (64 + 16 * wv) * W, tile_zero<W>());
    }
    if (it.y == IT_FDIAG) return;
    __syncthreads();
    for (int r0 = ne; r0 < m; r0 += SB) {
        const int nr = min(SB, m - r0);
        acc[0] = acc[1] = tile_zero<W>();
        fwd_rows<W, false>(L, lda, r0, nr, ne, nullptr, nq, acc, xo, S.err);
        store_rows(acc, r0, nr);
    }
    stores_done_barrier();
    if (tid == 0) publish_add(S.done + (size_t)grp * P.nfront + li);
}

// z = D^-1 y for column jj of a front (MixedDiagonal::solve_in_place, diagonal.rs:312-365):
// 1x1 -> y / d (0 for a zero pivot); a 2x2 by Cramer's rule (0 for a singular block).  y has row
// stride nq.
__device__ __forceinline__ double dsolve_col(const SolveFront &F, int jj, const double *__restrict__ y, int nq) {
    const int kd = gbl(F.dkind)[jj];
    if (kd == 1) {
        const double d = gbl(F.ddiag)[jj];
        return (d == 0.0) ? 0.0 : y[(size_t)jj * nq] / d;
    }
    const int f = (kd == 2) ? jj : jj - 1;  // first column of the 2x2
    const double a = gbl(F.ddiag)[f], b = gbl(F.doff)[f], cc = gbl(F.ddiag)[f + 1];
    const double det = a * cc - b * b;
    if (det == 0.0) return 0.0;
    const double r1 = y[(size_t)f * nq], r2 = y[(size_t)(f + 1) * nq];
    return (kd == 2) ? (cc * r1 - b * r2) / det : (a * r2 - b * r1) / det;
}

// ===========================================================================
// Backward sweep (one launch).
// ===========================================================================
template <int W>
__global__ __launch_bounds__(256, 2) void k_bwd_sweep(PlanDev P, const int4 *__restrict__ items, int nwork, int ngrp,
                                                      int nrhs, int wq, double *__restrict__ x, long long n,
                                                      const double *__restrict__ Wx, double *__restrict__ Xb,
                                                      long long wtotal, double *__restrict__ Pp, long long ptotal,
                                                      SyncDev S) {
    constexpr int NE = W / 4;
    const int t = take_ticket(S.tick + 1);
    if (t >= nwork) return;
    const int4 it = items[t / ngrp];
    const int grp = t % ngrp, q0 = grp * wq, nq = min(wq, nrhs - q0);
    const int li = it.x;
    const SolveFront &Fr = P.sf[li];
    const int ne = Fr.ne, m = Fr.m, r = m - ne;
    const size_t lda = (size_t)m;
    const gdouble *L = gbl(Fr.F);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int trow = tile_row(lane), qc = tile_col<W>(lane);
    const int nblk = (ne + SB - 1) / SB;
    const int fb = grp * P.nflag + Fr.fbase;
    const int nch = Fr.nchk;
    double *xg = x + (size_t)q0 * n;
    double *Pg = Pp + (size_t)q0 * ptotal;
    __shared__ __align__(16) double xs[2 * SB * W];
    __shared__ double frags[2 * TFRAG];
    static_assert(GH == 2 * SB, "a chunk's rows fill xs");
    // x of the L21 rows ne + rb .. ne + rb + nr - 1 into xs, zeros beyond (device-coherent:
    // ancestors write them in the same launch)
    auto gather = [&](int rb, int nr) {
        const gint *ri = gbl(Fr.sidx) + ne + rb;
        constexpr int NI = GH * W / 256;
        int g[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int e = tid + 256 * i, row = e / W;
            g[i] = (row < nr && e % W < nq) ? ri[row] : -1;
            if (g[i] >= n) {
                atomicOr(S.err, 2);  // an index outside the system: the solve plan does not fit the fronts
                g[i] = -1;
            }
        }
        double v[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) v[i] = g[i] >= 0 ? ld_co(xg + (size_t)g[i] * nq + (tid + 256 * i) % W) : 0.0;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int e = tid + 256 * i;
            xs[tcol_pos(e / W) * W + e % W] = v[i];
        }
    };
    TCols<W> T;
    // a chunk's first 128 rows ...
    auto chunk_start = [&](int rb, int nr, int c0, int ncols) {
        T.at(L, lda, ne + rb, min(SB, nr), c0, ncols);
        if (32 * wv < ncols) T.load_all();
    };
    // ... and the sum over the chunk for this wavefront's 32 columns
    auto chunk_sum = [&](int rb, int nr, int ncols) {
        Tile2<W> v{{tile_zero<W>(), tile_zero<W>()}};
        gather(rb, nr);
        __syncthreads();
        if (32 * wv < ncols) {
            v = T.step(xs, SB, max(nr - SB, 0));
            if (nr > SB) v = v + T.step(xs + SB * W, 0, 0);
        }
        return v;
    };
    // chunk items and fused fronts read the x of L21 rows: every ancestor has finished
    auto wait_parent = [&]() {
        if (tid == 0 && Fr.epar >= 0)
            wait_at_least(S.done + (size_t)grp * P.nfront + Fr.epar, Fr.epar_nblk, S.err);
        __syncthreads();
    };
    if (it.y == IT_BCHUNK) {
        const int C = it.z / nch, h = it.z % nch;
        const int c0 = C * SB, ncols = min(SB, ne - c0);
        const int rb = h * GH, nr = min(GH, r - rb);
        chunk_start(rb, nr, c0, ncols);
        wait_parent();
        const Tile2<W> v = chunk_sum(rb, nr, ncols);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                const int j = 32 * wv + 16 * tt + trow, q = qc + e;
                if (j < ncols && q < nq)
                    st_co(Pg + (size_t)(Fr.pbase + ((long long)C * nch + h) * SB + j) * nq + q, v.t[tt].e[e]);
            }
        stores_done_barrier();
        if (tid == 0) publish_add(S.bgc + fb + C);
        return;
    }
    // IT_BDIAG (column block C) or IT_BSMALL (the whole front, C = 0)
    const int C = it.z, j0 = C * SB;
    const int nb = min(SB, ne - j0);
    Diag<false, W == 4> dg;
    dg.load(L, lda, j0, nb, frags);
    int st[2];  // global indices of the rows this lane finishes
    Tile<W> acc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = 64 * h + 16 * wv + trow;
        st[h] = row < nb ? gbl(Fr.sidx)[j0 + row] : 0;
        const int col = 32 * wv + 16 * h + trow;
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int q = qc + e;
            acc[h].e[e] = (col < nb && q < nq)
                              ? dsolve_col(Fr, j0 + col, Wx + (size_t)q0 * wtotal + (size_t)Fr.wbase * nq + q, nq)
                              : 0.0;
        }
    }
    auto take_off = [&](const Tile2<W> &v) {
        acc[0] = acc[0] - v.t[0];
        acc[1] = acc[1] - v.t[1];
    };
    if (it.y == IT_BSMALL) {
        if (nch > 0) chunk_start(0, min(GH, r), 0, ne);
        wait_parent();
        // L21^T x_rows chunk by chunk, subtracted in chunk order (as the chunk partials are)
        for (int h = 0; h < nch; ++h) {
            const int rb = h * GH, nr = min(GH, r - rb);
            if (h > 0) chunk_start(rb, nr, 0, ne);
            take_off(chunk_sum(rb, nr, ne));
            __syncthreads();
        }
    } else if (r > 0) {
        if (tid == 0) wait_at_least(S.bgc + fb + C, nch, S.err);
        __syncthreads();
        for (int h = 0; h < nch; ++h) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int e = 0; e < NE; ++e) {
                    const int j = 32 * wv + 16 * tt + trow, q = qc + e;
                    if (j < nb && q < nq)
                        acc[tt].e[e] -= ld_co(Pg + (size_t)(Fr.pbase + ((long long)C * nch + h) * SB + j) * nq + q);
                }
        }
    }
    // later blocks of the same front, as they are published (descending), a whole tile of L in
    // flight ahead of the products
    if (nblk - 1 > C) {
        const double *Xf = Xb + (size_t)q0 * wtotal + (size_t)Fr.wbase * nq;
        const bool act = 32 * wv < nb;
        const int nr = ne - (nblk - 1) * SB;
        T.at(L, lda, (nblk - 1) * SB, nr, j0, nb);
        if (act) T.load_all();
        XBlock<W, true> X;
        if (X.AHEAD) X.ask(Xf + (size_t)(nblk - 1) * SB * nq, nr, nq);
        for (int Cp = nblk - 1; Cp > C; --Cp) {
            double *xb = xs + (Cp & 1) * (SB * W);
            if (!X.AHEAD) X.ask(Xf + (size_t)Cp * SB * nq, Cp == nblk - 1 ? nr : SB, nq);
            X.take(Cp <= C + NEAR, xb, S.err);
            if (X.AHEAD && Cp > C + 1) X.ask(Xf + (size_t)(Cp - 1) * SB * nq, SB, nq);
            if (act) take_off(T.step(xb, -SB, Cp > C + 1 ? SB : 0));
        }
    }
    if (W != 4 && dg.n2 > 0) dg.load_c(L, lda, j0);
    // The block's right-hand side, from which every later block and L21 have been removed, then its
    // x with L11^T.  The half of xs that the last block of x did not use is free.
    double *ws = xs + (C & 1) * (SB * W), *xo = xs + ((C + 1) & 1) * (SB * W);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) tile_store<W>(ws + (32 * wv + 16 * tt) * W, acc[tt]);
    __syncthreads();
    auto finish = [&](int h, int nn, const Tile<W> &v) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int row = 16 * wv + trow, q = qc + e;
            if (row < nn && q < nq) {
                if (nblk > 1)
                    publish_value(Xb + (size_t)q0 * wtotal + (size_t)(Fr.wbase + j0 + 64 * h + row) * nq + q, v.e[e]);
                if ((unsigned)st[h] < (unsigned)n) st_co(xg + (size_t)st[h] * nq + q, v.e[e]);
                else atomicOr(S.err, 2);
            }
        }
    };
    auto own = [&](int h) { return tile_load<W>(ws + (64 * h + 16 * wv) * W); };
    Tile<W> wa = own(0);
    if (dg.n2 > 0) {
        const Tile<W> xb = own(1) + dg.template tri_sum<W>(1, ws);
        tile_store<W>(xo + 16 * wv * W, xb);
        finish(1, dg.n2, xb);
        __syncthreads();
        // C^T x_B: 16 sums over four rows, added as a binary tree
        const double *xr = xo + (lane >> 4) * W + qc;
        wa = wa - tree_sum<16, Tile<W>>(0, [&](int s) {
                 Tile<W> p = tile_zero<W>();
                 mma<W>(dg.c[s], xr + 4 * s * W, p);
                 return p;
             });
        tile_store<W>(ws + 16 * wv * W, wa);
        __syncthreads();
    }
    finish(0, dg.n1, wa + dg.template tri_sum<W>(0, ws));
    stores_done_barrier();
    if (tid == 0) publish_add(S.done + (size_t)grp * P.nfront + li);
}

}  // namespace

void NumericGPU::prepare_solve() {
    const Prepared &P = *prep_;
    const int ns = (int)P.sns.size();
    const i64 n = P.n;
    // fronts taking part (ne > 0), in level order
    std::vector<int> flist, li_of(ns, -1);
    for (const auto &lv : P.levels)
        for (int s : lv)
            if (ne_[s] > 0) {
                li_of[s] = (int)flist.size();
                flist.push_back(s);
            }
    const int nf = (int)flist.size();
    // per-front bases
    std::vector<long long> wb(nf), yb(nf), pb(nf);
    std::vector<int> fbase(nf), nrow(nf), nchk(nf);
    std::vector<long long> ybase_sn(ns, 0);
    long long wt = 0, yt = 0, pt = 0;
    int nflag = 0;
    for (int li = 0; li < nf; ++li) {
        const int s = flist[li];
        const int ne = ne_[s], r = m_[s] - ne, nblk = (ne + SB - 1) / SB;
        wb[li] = wt;
        wt += ne;
        yb[li] = yt;
        ybase_sn[s] = yt;
        yt += r;
        fbase[li] = nflag;
        nflag += nblk;
        nrow[li] = (r + SB - 1) / SB;
        nchk[li] = (r + GH - 1) / GH;
        pb[li] = pt;
        pt += (long long)nblk * nchk[li] * SB;
    }
    // pull lists: for each global index, the Y entries of the fronts (postorder) that update it
    std::vector<int> cnt(n + 1, 0);
    for (int s = 0; s < ns; ++s) {
        if (ne_[s] == 0) continue;
        for (int g : delayed_[s]) cnt[g + 1]++;
        for (int g : P.sns[s].pattern) cnt[g + 1]++;
    }
    for (i64 i = 0; i < n; ++i) cnt[i + 1] += cnt[i];
    std::vector<long long> ent(cnt[n]);
    {
        std::vector<int> pos(cnt.begin(), cnt.end() - 1);
        for (int s = 0; s < ns; ++s) {
            if (ne_[s] == 0) continue;
            long long p = ybase_sn[s];
            for (int g : delayed_[s]) ent[pos[g]++] = p++;
            for (int g : P.sns[s].pattern) ent[pos[g]++] = p++;
        }
    }
    // unresolved columns (delays left at the roots)
    std::vector<int> unres;
    for (int s = 0; s < ns; ++s)
        if (P.sns[s].parent < 0) unres.insert(unres.end(), delayed_[s].begin(), delayed_[s].end());
    // effective children / parent: nearest descendants (ancestor) with ne > 0
    auto fused = [&](int li) {
        const int s = flist[li];
        return ne_[s] <= SB && m_[s] - ne_[s] <= FUSE_R;
    };
    std::vector<int> ech_ptr(nf + 1, 0), echf, epar(nf, -1);
    for (int li = 0; li < nf; ++li) {
        std::vector<int> stack(P.children[flist[li]].rbegin(), P.children[flist[li]].rend());
        while (!stack.empty()) {
            const int c = stack.back();
            stack.pop_back();
            if (ne_[c] > 0) {
                echf.push_back(li_of[c]);
                epar[li_of[c]] = li;
            } else {
                stack.insert(stack.end(), P.children[c].rbegin(), P.children[c].rend());
            }
        }
        ech_ptr[li + 1] = (int)echf.size();
    }
    // forward done target of a front: its rows items, or 1 for a fused front
    auto ndone = [&](int li) { return fused(li) ? 1 : nrow[li]; };
    std::vector<int2> ech(echf.size());
    for (size_t e = 0; e < echf.size(); ++e) ech[e] = make_int2(echf[e], ndone(echf[e]));
    std::vector<SolveFront> sf(nf);
    for (int li = 0; li < nf; ++li) {
        const int s = flist[li];
        const FrontDev &h = h_fr_[s];
        SolveFront &f = sf[li];
        f.F = h.Lf;
        f.sidx = h.sidx;
        f.dkind = h.dkind;
        f.ddiag = h.ddiag;
        f.doff = h.doff;
        f.wbase = wb[li];
        f.ybase = yb[li];
        f.pbase = pb[li];
        f.m = m_[s];
        f.ne = ne_[s];
        f.fbase = fbase[li];
        f.nchk = nchk[li];
        f.ech0 = ech_ptr[li];
        f.ech1 = ech_ptr[li + 1];
        f.epar = epar[li];
        f.epar_nblk = epar[li] >= 0 ? ndone(epar[li]) + (ne_[flist[epar[li]]] + SB - 1) / SB : 0;
    }
    // items: forward by levels bottom-up, backward top-down.  Within a level: forward, the
    // diagonal (and fused) items by block step across fronts, then the rows items; backward, the
    // fused and chunk items, then the diagonal items by step (last block first).
    std::vector<int4> fit, bit;
    std::vector<std::vector<int>> lvl_fronts(P.levels.size());
    for (size_t lv = 0; lv < P.levels.size(); ++lv)
        for (int s : P.levels[lv])
            if (ne_[s] > 0) lvl_fronts[lv].push_back(li_of[s]);
    auto nblk_of = [&](int li) { return (ne_[flist[li]] + SB - 1) / SB; };
    for (size_t lv = 0; lv < lvl_fronts.size(); ++lv) {
        const auto &fl = lvl_fronts[lv];
        int maxblk = 0;
        for (int li : fl) maxblk = std::max(maxblk, nblk_of(li));
        for (int c = 0; c < maxblk; ++c)
            for (int li : fl)
                if (c < nblk_of(li)) fit.push_back(make_int4(li, fused(li) ? IT_FSMALL : IT_FDIAG, c, 0));
        for (int li : fl)
            if (!fused(li))
                for (int g = 0; g < nrow[li]; ++g) fit.push_back(make_int4(li, IT_FROWS, g, 0));
    }
    for (int lv = (int)lvl_fronts.size() - 1; lv >= 0; --lv) {
        const auto &fl = lvl_fronts[lv];
        int maxblk = 0;
        for (int li : fl) {
            if (fused(li)) {
                bit.push_back(make_int4(li, IT_BSMALL, 0, 0));
                continue;
            }
            maxblk = std::max(maxblk, nblk_of(li));
            for (int C = nblk_of(li) - 1; C >= 0; --C)
                for (int h = 0; h < nchk[li]; ++h) bit.push_back(make_int4(li, IT_BCHUNK, C * nchk[li] + h, 0));
        }
        for (int step = 0; step < maxblk; ++step)
            for (int li : fl)
                if (!fused(li) && step < nblk_of(li)) bit.push_back(make_int4(li, IT_BDIAG, nblk_of(li) - 1 - step, 0));
    }
    // diagonal triangles (64 columns each) of every front, inverted after each factorization;
    // grouped by order class (<= 16, <= 32, <= 64), one launch per class
    std::vector<int4> tcls[3], tris;
    for (int li = 0; li < nf; ++li) {
        const int ne = ne_[flist[li]];
        for (int jb = 0; jb < ne; jb += 64) {
            const int tn = std::min(64, ne - jb);
            tcls[tn <= 16 ? 0 : tn <= 32 ? 1 : 2].push_back(make_int4(li, jb, tn, 0));
        }
    }
    for (int c = 0; c < 3; ++c) {
        sm_.ntri[c] = (int)tcls[c].size();
        tris.insert(tris.end(), tcls[c].begin(), tcls[c].end());
    }
    // device metadata
    std::vector<char> &st = sol_meta_host_;
    st.clear();
    auto push = [&](const void *p, size_t bytes) {
        size_t off = (st.size() + 255) / 256 * 256;
        st.resize(off + std::max<size_t>(bytes, 1));
        if (bytes) std::memcpy(st.data() + off, p, bytes);
        return off;
    };
    const size_t o_ptr = push(cnt.data(), cnt.size() * sizeof(int));
    const size_t o_ent = push(ent.data(), ent.size() * sizeof(long long));
    const size_t o_sf = push(sf.data(), sf.size() * sizeof(SolveFront));
    const size_t o_ec = push(ech.data(), ech.size() * sizeof(int2));
    const size_t o_fit = push(fit.data(), fit.size() * sizeof(int4));
    const size_t o_bit = push(bit.data(), bit.size() * sizeof(int4));
    const size_t o_un = push(unres.data(), unres.size() * sizeof(int));
    const size_t o_tr = push(tris.data(), tris.size() * sizeof(int4));
    if (st.size() > sol_meta_bytes_) {
        if (d_sol_meta_) (void)hipFree(d_sol_meta_);
        d_sol_meta_ = nullptr;
        sol_meta_bytes_ = 0;
        RV_HIP(hipMalloc(&d_sol_meta_, st.size()));
        sol_meta_bytes_ = st.size();
    }
    RV_HIP(hipMemcpy(d_sol_meta_, st.data(), st.size(), hipMemcpyHostToDevice));
    char *b = (char *)d_sol_meta_;
    sm_.ptr = (const int *)(b + o_ptr);
    sm_.ent = (const long long *)(b + o_ent);
    sm_.fronts = (const void *)(b + o_sf);
    sm_.ech = (const int2 *)(b + o_ec);
    sm_.fitems = (const int4 *)(b + o_fit);
    sm_.bitems = (const int4 *)(b + o_bit);
    sm_.nfitems = (int)fit.size();
    sm_.nbitems = (int)bit.size();
    sm_.unres = (const int *)(b + o_un);
    sm_.tris = (const int4 *)(b + o_tr);
    sm_.ntris = (int)tris.size();
    inv_valid_ = false;
    sm_.nunres = (int)unres.size();
    sm_.nfront = nf;
    sm_.nflag = nflag;
    sm_.wtotal = std::max<long long>(wt, 1);
    sm_.ytotal = std::max<long long>(yt, 1);
    sm_.ptotal = std::max<long long>(pt, 1);
    sol_plan_gen_ = plan_gen_;
    solve_ready_ = true;
}

// Columns per group of right-hand sides, dealt evenly to groups of at most 4 or, past 32 columns,
// 8.  Groups of 4 have the shorter chain step, groups of 8 read the factor half as often, which
// counts once the groups fill the chip.  How many groups do depends on the factor; the line is that of
// Helmholtz 40^3, between the small factors, whose groups of 4 stay ahead throughout, and the large
// ones, whose groups of 8 lead from 12 to 20 columns on.  Both sweeps, groups of at most 4 / of 8, us:
//   columns                 8            16            32            64
//   Helmholtz 20^3     270 /  346    269 /  355    288 /  358    345 /  384
//   KKT side 64        489 /  685    517 /  698    584 /  720    684 /  800
//   KKT side 128      3820 / 5860   4080 / 5890   4640 / 6220   6140 / 7040
//   Helmholtz 40^3     657 /  875    819 /  967   1170 / 1170   1980 / 1630
//   2-D grid 400^2     937 /  810   1560 / 1190   2930 / 2050   5780 / 3850
//   48 KKT systems    1615 / 1588   2550 / 2135   4500 / 3330   8440 / 5860
//   Helmholtz 64^3    2570 / 2700   3770 / 3410   6330 / 4930  11600 / 8260
int NumericGPU::solve_group_width(int nrhs) {
    if (nrhs <= 0) return 1;
    const int most = nrhs <= 32 ? 4 : 8;
    const int ngrp = (nrhs + most - 1) / most;
    return (nrhs + ngrp - 1) / ngrp;
}

long long NumericGPU::solve_scratch_bytes(int nrhs) const {
    const int nr = solve_group_width(nrhs);
    const long long ngrp = nrhs > 0 ? (nrhs + nr - 1) / nr : 0;
    const long long nsync = 2 + 1 + ngrp * ((long long)sm_.nflag + sm_.nfront);
    const long long doubles = ((long long)prep_->n + 2 * sm_.wtotal + sm_.ytotal + sm_.ptotal) * nrhs;
    return ((doubles * 8 + 255) / 256) * 256 + ((nsync * 4 + 255) / 256) * 256;
}

void NumericGPU::solve(double *d_rhs, i64 ldrhs, int nrhs, const double *d_scaling) {
    if (!solve_ready_) prepare_solve();
    const i64 n = prep_->n;
    if (n == 0 || nrhs <= 0) return;
    void *ws = sol_buf_.get((size_t)solve_scratch_bytes(nrhs));
    solve_with(d_rhs, ldrhs, nrhs, d_scaling, ws);
    int err = 0;
    RV_HIP(hipMemcpyAsync(&err, sol_err_, sizeof(int), hipMemcpyDeviceToHost, stream_));
    RV_HIP(hipStreamSynchronize(stream_));
    if (err) throw std::runtime_error(solve_error_text(err));
}

// The solve on a caller-provided workspace of solve_scratch_bytes(nrhs) bytes (device memory,
// 256-byte aligned), enqueued on the library stream; allocates nothing.  The error word (set
// when a dependency wait exceeded its limit) is left at sol_err_.
void NumericGPU::solve_with(double *d_rhs, i64 ldrhs, int nrhs, const double *d_scaling, void *work) {
    const Prepared &P = *prep_;
    const i64 n = P.n;
    const int wq = solve_group_width(nrhs);
    const int ngrp = (nrhs + wq - 1) / wq;
    const long long wt = sm_.wtotal, yt = sm_.ytotal, pt = sm_.ptotal, nn = n;
    double *xp = (double *)work;
    double *W = xp + (size_t)n * nrhs;
    double *Xb = W + (size_t)wt * nrhs;
    double *Y = Xb + (size_t)wt * nrhs;
    double *Pp = Y + (size_t)yt * nrhs;
    const long long doubles = ((long long)n + 2 * wt + yt + pt) * nrhs;
    int *sync = (int *)((char *)work + ((doubles * 8 + 255) / 256) * 256);
    const long long nsync = 3 + (long long)ngrp * ((long long)sm_.nflag + sm_.nfront);
    SyncDev S;
    S.tick = sync;
    S.err = sync + 2;
    S.bgc = sync + 3;
    S.done = S.bgc + (size_t)ngrp * sm_.nflag;
    sol_err_ = S.err;
    PlanDev D;
    D.sf = (const SolveFront *)sm_.fronts;
    D.ech = sm_.ech;
    D.ptr = sm_.ptr;
    D.ent = sm_.ent;
    D.nfront = sm_.nfront;
    D.nflag = sm_.nflag;
    if (!inv_valid_) {
        // the first solve after a factorization inverts the diagonal triangles
        const int4 *tp = sm_.tris;
        if (sm_.ntri[0] > 0)
            hipLaunchKernelGGL(k_diag_inverse<16>, dim3((unsigned)sm_.ntri[0]), dim3(64), 0, stream_,
                               (const SolveFront *)sm_.fronts, tp);
        tp += sm_.ntri[0];
        if (sm_.ntri[1] > 0)
            hipLaunchKernelGGL(k_diag_inverse<32>, dim3((unsigned)sm_.ntri[1]), dim3(64), 0, stream_,
                               (const SolveFront *)sm_.fronts, tp);
        tp += sm_.ntri[1];
        if (sm_.ntri[2] > 0)
            hipLaunchKernelGGL(k_diag_inverse<64>, dim3((unsigned)sm_.ntri[2]), dim3(64), 0, stream_,
                               (const SolveFront *)sm_.fronts, tp);
        inv_valid_ = true;
    }
    const dim3 gn((unsigned)((n + 255) / 256), (unsigned)ngrp);
    hipLaunchKernelGGL(k_solve_start, gn, dim3(256), 0, stream_, d_rhs, (long long)ldrhs, xp, nn, nrhs, wq,
                       P.d_perm_fwd, d_scaling, sync, nsync, (unsigned long long *)W, 2 * wt * nrhs);
    const int nfw = sm_.nfitems * ngrp, nbw = sm_.nbitems * ngrp;
    if (nfw > 0)
        hipLaunchKernelGGL((wq <= 4 ? k_fwd_sweep<4> : k_fwd_sweep<8>), dim3((unsigned)nfw), dim3(256), 0, stream_, D,
                           sm_.fitems, nfw, ngrp, nrhs, wq, (const double *)xp, nn, W, wt, Y, yt, S);
    if (sm_.nunres > 0)
        hipLaunchKernelGGL(k_pull_rows, dim3((sm_.nunres + 255) / 256, nrhs), dim3(256), 0, stream_, sm_.unres,
                           sm_.nunres, sm_.ptr, sm_.ent, (const double *)Y, yt, xp, nn, nrhs, wq);
    if (nbw > 0)
        hipLaunchKernelGGL((wq <= 4 ? k_bwd_sweep<4> : k_bwd_sweep<8>), dim3((unsigned)nbw), dim3(256), 0, stream_, D,
                           sm_.bitems, nbw, ngrp, nrhs, wq, xp, nn, (const double *)W, Xb, wt, Pp, pt, S);
    hipLaunchKernelGGL(k_perm_out, gn, dim3(256), 0, stream_, d_rhs, (long long)ldrhs, (const double *)xp, nn, nrhs,
                       wq, P.d_perm_fwd, d_scaling);
}

// ===========================================================================
// Fixed workspace of the allocation-free solve entry point: one array per GPU, held until the
// process ends.  Host code never passes the array's name to a kernel (on the host it names a
// stand-in, not device memory): the device address comes from hipGetSymbolAddress, once per
// device, with that device current.
// ===========================================================================
namespace {
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)RV_SOLVE_NOALLOC_BYTES;
__device__ __align__(256) char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[MAX_DEVICES] = {};
}  // namespace

size_t noalloc_scratch_bytes() { return NOALLOC_SCRATCH_BYTES; }

std::string solve_error_text(int err) {
    std::string m = "solve failed, results invalid:";
    if (err & 1) m += " a dependency wait exceeded its limit;";
    if (err & 2) m += " an index fell outside the system (solve plan and fronts disagree);";
    return m;
}

void *noalloc_scratch() {
    int dev = 0;
    RV_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= MAX_DEVICES) throw std::runtime_error("device index beyond the supported range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        RV_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) throw std::runtime_error("hipGetSymbolAddress returned no address for the solve workspace");
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

}  // namespace rv
