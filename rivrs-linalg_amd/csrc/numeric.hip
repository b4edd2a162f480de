// numeric.hip -- MI355X (gfx950) numeric factorization of the multifrontal APTP LDL^T.
//
// Fronts are processed level by level of the assembly tree (leaves first), all fronts of a
// level in the same launches.  Per level:
//   1. assembly      k_scatter_orig (original entries) + k_extend_add (one launch per round of
//                    children without common rows, so a parent's entries sum their children in
//                    reference order)
//   2. dense factor  fronts with k < ib or inside a small-leaf subtree: k_tpp (threshold
//                    partial pivoting, one workgroup per front);
//                    other fronts: APTP with ib x ib complete pivoting blocks
//                    (k_block_apply -> k_block_update -> k_block_finish per inner block, the
//                    trailing update restricted to the outer block, and the rank-nb outer
//                    update k_form_ld + k_schur on MFMA), then k_tpp on the columns APTP left.
//   3. contribution  k_form_ld + k_schur: C -= (L21 D) L21^T on the NFS x NFS block, FP64 MFMA.
//   4. k_collect     eliminated counts, D inertia and delayed columns for the host.
// The host plans every level from the children's results the previous factorization
// produced and enqueues all levels without waiting; levels above one whose delays differ
// from that plan are planned again and rerun (NumericGPU::factor).
// The scalar pivoting arithmetic is compiled without FMA contraction so that every decision
// step reproduces the reference's operation sequence (sparse/src/symmetric/factor.rs).
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "rv_numeric.h"

namespace rv {

// ===========================================================================
// Arena / buffers
// ===========================================================================
void *DevArena::alloc(size_t bytes, size_t align) {
    bytes = (bytes + align - 1) / align * align;
    if (bytes == 0) bytes = align;
    while (cur_ < chunks_.size()) {
        Chunk &c = chunks_[cur_];
        const size_t off = (c.used + align - 1) / align * align;
        if (off + bytes <= c.size) {
            c.used = off + bytes;
            return c.base + off;
        }
        if (cur_ + 1 >= chunks_.size()) break;
        chunks_[++cur_].used = 0;
    }
    const size_t sz = std::max(bytes, (size_t)256 << 20);
    void *p = nullptr;
    RV_HIP(hipMalloc(&p, sz));
    chunks_.push_back(Chunk{(char *)p, sz, bytes});
    cur_ = chunks_.size() - 1;
    reserved_ += sz;
    return p;
}

void DevArena::reset_keep() {
    cur_ = 0;
    if (!chunks_.empty()) chunks_[0].used = 0;
}

DevArena::Mark DevArena::mark() const {
    Mark m;
    m.chunk = cur_;
    m.used = cur_ < chunks_.size() ? chunks_[cur_].used : 0;
    return m;
}

void DevArena::reset_to(const Mark &m) {
    cur_ = m.chunk;
    if (cur_ < chunks_.size()) chunks_[cur_].used = m.used;
}

void DevArena::release() {
    for (Chunk &c : chunks_) (void)hipFree(c.base);
    chunks_.clear();
    cur_ = 0;
    reserved_ = 0;
}

void *DevBuf::get(size_t bytes) {
    if (bytes <= cap && p) return p;
    if (p) (void)hipFree(p);
    cap = std::max(bytes, cap * 3 / 2);
    cap = std::max(cap, (size_t)4096);
    RV_HIP(hipMalloc(&p, cap));
    return p;
}

DevBuf::~DevBuf() {
    if (p) (void)hipFree(p);
}

void FrontPool::reserve(size_t bytes) {
    if (virtual_ || !chunks_.empty() || bytes == 0) return;
    bytes = (bytes + 255) / 256 * 256;
    void *p = nullptr;
    RV_HIP(hipMalloc(&p, bytes));
    chunks_.push_back(Chunk{(char *)p, bytes});
    reserved_ += bytes;
}

void FrontPool::drop_from(int lv) {
    size_t n = 0;
    for (const Block &b : blocks_)
        if (b.lv < lv) blocks_[n++] = b;
    blocks_.resize(n);
}

int FrontPool::place(int lv, int death, size_t bytes) {
    bytes = std::max<size_t>((bytes + 255) / 256 * 256, 256);
    if (virtual_ && chunks_.empty()) chunks_.push_back(Chunk{nullptr, SIZE_MAX});
    std::vector<std::pair<size_t, size_t>> iv;
    for (size_t c = 0; c <= chunks_.size(); ++c) {
        if (c == chunks_.size()) {
            // no chunk has room: a new one (its blocks are placed from its start)
            const size_t sz = std::max(bytes, (size_t)256 << 20);
            void *p = nullptr;
            RV_HIP(hipMalloc(&p, sz));
            chunks_.push_back(Chunk{(char *)p, sz});
            reserved_ += sz;
        }
        iv.clear();
        for (const Block &b : blocks_)
            if (b.chunk == (int)c && (b.lv == lv || (b.lv < lv && b.death >= lv)))
                iv.emplace_back(b.off, b.off + b.size);
        std::sort(iv.begin(), iv.end());
        size_t pos = 0;
        for (const auto &r : iv) {
            if (r.first >= pos + bytes) break;
            pos = std::max(pos, r.second);
        }
        if (pos + bytes > chunks_[c].size) continue;
        for (Block &b : blocks_)
            if (b.chunk == (int)c && b.lv < lv && b.death < lv && b.off < pos + bytes && pos < b.off + b.size)
                b.clobbered = true;
        blocks_.push_back(Block{(int)c, pos, bytes, lv, death, false});
        top_ = std::max(top_, pos + bytes);
        return (int)blocks_.size() - 1;
    }
    return -1;  // not reached
}

void FrontPool::release() {
    if (!virtual_)
        for (Chunk &c : chunks_) (void)hipFree(c.base);
    chunks_.clear();
    blocks_.clear();
    top_ = 0;
    reserved_ = 0;
}

// Phase timing of the inner-block kernels for a probe build (-DRV_PHASE_TIMING): workgroup 0,
// thread 0 of every launch adds the cycles since kernel start at each phase mark.
#ifdef RV_PHASE_TIMING
__device__ unsigned long long g_phase[2][16];
__device__ unsigned long long g_phase_launches[2];
#define RV_PHASE_START() const unsigned long long rv_t0_ = clock64()
#define RV_PHASE(kern, i)                                                              \
    do {                                                                               \
        if (blockIdx.x == 0 && threadIdx.x == 0)                                       \
            atomicAdd(&g_phase[kern][i], (unsigned long long)(clock64() - rv_t0_));     \
    } while (0)
#define RV_PHASE_COUNT(kern)                                                           \
    do {                                                                               \
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&g_phase_launches[kern], 1ull); \
    } while (0)
#else
#define RV_PHASE_START() do {} while (0)
#define RV_PHASE(kern, i) do {} while (0)
#define RV_PHASE_COUNT(kern) do {} while (0)
#endif

// ===========================================================================
// Device helpers
// ===========================================================================
__device__ __forceinline__ bool aptp_active(int p, int nb, int ib, int ob, int it) {
    const bool two = p > nb;
    const int nouter = two ? (p + nb - 1) / nb : 1;
    if (ob >= nouter) return false;
    const int obcols = two ? min(nb, p - ob * nb) : p;
    return it < (obcols + ib - 1) / ib;
}

__device__ __forceinline__ double wave_fmax(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

__device__ __forceinline__ int wave_min_int(int v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return v;
}

__device__ __forceinline__ void atomic_max_nonneg(unsigned long long *p, double v) {
    if (v > 0.0) atomicMax(p, (unsigned long long)__double_as_longlong(v));
}

// effective nelim of an inner block: first failing pivot, never splitting a 2x2
// (apply_and_check + adjust_for_2x2_boundary, factor.rs:1160-1172, 1295-1408)
__device__ __forceinline__ int effective_nelim(const AptpState &S) {
    int e = min(S.fail_min, S.block_nelim);
    if (e > 0 && S.bkind[e - 1] == 2) e -= 1;
    return e;
}

// W = L * D entry (compute_ld_into, factor.rs:1536-1563) for row values of the pivot columns.
// kind: 1 = 1x1, 2 = first of 2x2, 3 = second of 2x2.
template <class P>
__device__ __forceinline__ double ld_entry(P rowbase, size_t lda, int c, int kind, const double *diag,
                                           const double *off) {
    if (kind == 1) return rowbase[c * lda] * diag[c];
    if (kind == 2) {
        const double l1 = rowbase[c * lda], l2 = rowbase[(c + 1) * lda];
        return l1 * diag[c] + l2 * off[c];
    }
    if (kind == 3) {
        const double l1 = rowbase[(c - 1) * lda], l2 = rowbase[c * lda];
        return l1 * off[c - 1] + l2 * diag[c];
    }
    return 0.0;
}

// ===========================================================================
// Assembly
// ===========================================================================
struct ScatterChunk { int front; int begin; int end; int pad; };

// Fronts are zeroed in their lower triangle only (diagonal included): every kernel reads and
// writes only that part of a front.  Work item (front, ZCOLS columns), one column at a time.
constexpr int ZCOLS = 16;

// A level's set-up in one launch (the parts are independent; descriptors are read from the
// level's staged copy lfr): workgroups [0, nzl) zero the fronts' lower triangles (ZCOLS columns
// each), the next cdiv(nf, 256) install the descriptors, the next nf set perm = identity, the
// rest copy the level's row lists (1024 entries each).
constexpr int ROWCOPY = 1024;
__global__ __launch_bounds__(256) void k_level_setup(FrontDev *__restrict__ fr, const int *__restrict__ ids,
                                                     const FrontDev *__restrict__ lfr, int nf,
                                                     const int2 *__restrict__ zitems, int nzl,
                                                     int *__restrict__ rows_dst, const int *__restrict__ rows_src,
                                                     long long nrows) {
    int b = blockIdx.x;
    const int tid = threadIdx.x;
    if (b < nzl) {
        const int2 it = zitems[b];
        const FrontDev &F = lfr[it.x];
        const int m = F.m;
        gdouble *A = gbl(F.F);
        const int c1 = min(it.y + ZCOLS, m);
        for (int c = it.y; c < c1; ++c)
            for (int r = c + tid; r < m; r += 256) A[r + (size_t)c * m] = 0.0;
        return;
    }
    b -= nzl;
    const int nset = (nf + 255) / 256;
    if (b < nset) {
        const int i = b * 256 + tid;
        if (i < nf) fr[ids[i]] = lfr[i];
        return;
    }
    b -= nset;
    if (b < nf) {
        const FrontDev &F = lfr[b];
        for (int i = tid; i < F.m; i += 256) gbl(F.perm)[i] = i;
        return;
    }
    b -= nf;
    const long long i0 = (long long)b * ROWCOPY;
    for (int u = tid; u < ROWCOPY; u += 256)
        if (i0 + u < nrows) rows_dst[i0 + u] = rows_src[i0 + u];
}

// Original entries (numeric.rs:1306-1344; fallback scatter numeric.rs:2376-2435 when delayed
// columns shift the pattern rows).  The two reference paths scale as (v*s_r)*s_c and
// v*(s_r*s_c) respectively; both are reproduced.
__global__ __launch_bounds__(256) void k_scatter_orig(const FrontDev *__restrict__ fr,
                                                      const ScatterChunk *__restrict__ ch,
                                                      const AmapEntry *__restrict__ amap,
                                                      const double *__restrict__ val,
                                                      const double *__restrict__ sc) {
    const ScatterChunk c = ch[blockIdx.x];
    const int e = c.begin + threadIdx.x;
    if (e >= c.end) return;
    const FrontDev &F = fr[c.front];
    const AmapEntry a = amap[e];
    int r = (int)a.row, col = (int)a.col;
    if (r >= F.n_owned) r += F.ndelay_in;
    if (col >= F.n_owned) col += F.ndelay_in;
    double v = val[a.src];
    if (sc) v = (F.ndelay_in == 0) ? (v * sc[a.sr]) * sc[a.sc] : v * (sc[a.sr] * sc[a.sc]);
    gbl(F.F)[r + (size_t)col * F.m] += v;
}

// Extend-add of one 64x64 lower tile of a child's contribution block (the trailing
// (m-ne)^2 block of the child front) into the parent, with both index maps staged in LDS
// (extend_add numeric.rs:2445-2485, extend_add_mapped 2507-2549).
__global__ __launch_bounds__(256) void k_extend_add(const FrontDev *__restrict__ fr,
                                                    const EaItem *__restrict__ items) {
    const EaItem it = items[blockIdx.x];
    const FrontDev &C = fr[it.child];
    const FrontDev &P = fr[it.parent];
    const int ne = it.cne;  // the child's eliminated count the parent's map was built for
    const int sz = C.m - ne;
    const size_t ldc = C.m;
    const gdouble *CB = gbl(C.F) + ne + (size_t)ne * ldc;
    const int i0 = it.ti * 64, j0 = it.tj * 64;
    __shared__ unsigned mi[64], mj[64];
    const int t = threadIdx.x;
    if (t < 64) mi[t] = (i0 + t < sz) ? gbl(it.map)[i0 + t] : 0u;
    else if (t < 128) mj[t - 64] = (j0 + t - 64 < sz) ? gbl(it.map)[j0 + t - 64] : 0u;
    __syncthreads();
    const int ii = t & 63;
    const int i = i0 + ii;
    if (i >= sz) return;
    gdouble *PF = gbl(P.F);
    const size_t ldp = P.m;
    // all loads first (the 16 targets of a thread are distinct), then the stores
    double v[16], pv[16];
    size_t dst[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int jj = (t >> 6) + 4 * u;
        const int j = j0 + jj;
        const bool ok = j < sz && i >= j;
        v[u] = ok ? CB[i + (size_t)j * ldc] : 0.0;
        const unsigned li = mi[ii], lj = mj[jj];
        dst[u] = (li >= lj) ? li + (size_t)lj * ldp : lj + (size_t)li * ldp;
        pv[u] = ok ? PF[dst[u]] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int j = j0 + (t >> 6) + 4 * u;
        if (j >= sz || i < j) continue;
        if (it.skip_zero && v[u] == 0.0) continue;
        PF[dst[u]] = pv[u] + v[u];
    }
}

// ===========================================================================
// Wavefront primitives.  DPP moves within rows of 16 lanes plus four readlanes reduce a
// wavefront without the LDS crossbar; callers keep all 64 lanes active.
// ===========================================================================
// Workgroup barrier that orders LDS only: global loads and stores in flight are not waited for.
__device__ __forceinline__ void lds_barrier() {
#ifdef RV_DBG_FULLBAR
    __syncthreads();
#else
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#endif
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    // every lane is written (full row and bank masks), so no old value is needed
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// fmax over the wavefront (NaN inputs are ignored, as by fmax)
__device__ __forceinline__ double wave_max_dpp(double v) {
    v = fmax(v, dpp_f64<0xB1>(v));   // quad_perm [1,0,3,2]
    v = fmax(v, dpp_f64<0x4E>(v));   // quad_perm [2,3,0,1]
    v = fmax(v, dpp_f64<0x141>(v));  // row_half_mirror
    v = fmax(v, dpp_f64<0x140>(v));  // row_mirror
    return fmax(fmax(readlane_f64(v, 0), readlane_f64(v, 16)),
                fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// Copy of the lower diagonal block [kpos, kpos + bs) of the next inner block (all threads of
// the calling workgroup).  Every workgroup of k_block_apply stages the block from this copy,
// because the first of them writes the factored block back into the front.
__device__ __forceinline__ void copy_next_block(const FrontDev &F, const AptpState &S, int ib) {
    const int k = S.kpos, bs = min(S.end_pos - k, ib);
    const size_t lda = F.m;
    for (int e = threadIdx.x; e < MAX_IB * MAX_IB; e += blockDim.x) {
        const int i = e & (MAX_IB - 1), j = e / MAX_IB;
        if (i < bs && j <= i) gbl(S.blkcopy)[e] = gbl(F.F)[(k + i) + (size_t)(k + j) * lda];
    }
}

// A value the compiler has to take as new: address arithmetic formed from it is neither hoisted
// out of the block loop nor kept from one phase to the next.  (Left to itself the compiler holds
// some hundred loop-invariant offsets of the unrolled loads and stores below in registers across
// the loop and spills the data instead: 440 spilled registers, 39 us per substitution.)
__device__ __forceinline__ int fresh(int x) {
    __asm__ volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ int fresh_uniform(int x) {
    x = __builtin_amdgcn_readfirstlane(x);
    __asm__ volatile("" : "+s"(x));
    return x;
}

// ===========================================================================
// APTP: complete pivoting on the inner block (factor_block_diagonal, factor.rs:891-1153).
// Returns the eliminated count; bp/bkind/bdiag/boff describe the pivots and *maxl the largest
// |l| of the block.
//
// The pivot steps are one serial chain, so one wavefront (the workgroup's first; the others wait
// at the closing barrier) runs them without any barrier, and everything is laid out for the
// fewest instructions and LDS round trips per step:
//  * The block is symmetric; every unordered pair {i, i + d mod 32}, d = 1 .. 16, has one owner.
//    Lane (i = lane & 31, h = lane >> 5) keeps e[u] = a(i, j), j = i + 1 + u + 8h (mod 32), in
//    registers: eight entries per lane with no lane idle (d = 16 would be owned twice; the copy
//    of the rows i >= 16 is dead), and the diagonal in lanes h = 0.
//  * Entries stay at their original indices; no row or column is moved.  pos[i] is the position
//    the reference's swaps would have put row i at.  It only decides the order of the factors of
//    an update (the row at the larger position gives l, the other w = l d) and ties.
//  * A dead entry (eliminated, outside the block, the second copy) is NaN.  fmax ignores it, the
//    diagonal of the LDS copy is NaN, so a pivot's own row gets NaN multipliers and dies in the
//    ordinary update: no masks.
//  * Argmax: an entry's key is the high word of its magnitude with the column index in the low
//    five bits; as a float its NaN is ignored and its order is the magnitudes'.  From 2^1017 on a
//    key would be a float NaN itself, which is why blocks with entries of 2^1000 or more always take
//    the exact rule.  (Looked at once, before the first pivot: a pivot is at least 1/sqrt 2 of the
//    largest entry left, a 2x2's determinant half its square, so by Hadamard's inequality, as in
//    Wilkinson's bound for complete pivoting, the entries of 32 columns grow by less than 2^11.)  Keys are reduced by v_max3 and
//    DPP, so the winner's row is its lane and its column the key's low bits.  It stands if no
//    other lane's key and no other entry of its row reaches its leading 15 mantissa bits;
//    otherwise (near-equal values, ties, tiny values) the exact rule runs: largest value, then
//    first in the column-major order of positions.
//  * A full symmetric copy of the block in LDS gives a lane the pivot row's entries of its own row
//    and of its eight columns in one round trip, beside the reciprocal of the pivot.
// A wavefront issues an operation every 5 to 6 cycles here (8 to 9 when it depends on the one
// before), an LDS round trip takes 70, a DPP stage 17, a division 76: a step with a diagonal
// winner is some 190 operations, 1320 cycles.  A 32-column block takes 18 us with diagonal
// winners and 23 us with entries of random signs and sizes, 25 us before the argmax worked on
// keys, 40 us as 256 threads with four entries each, one barrier per step and the block permuted
// through LDS.
// ===========================================================================
// max(|a|, |b|), NaN operands ignored (the compiler's fmax canonicalises loop-carried operands
// first, one more instruction each)
__device__ __forceinline__ double max_abs(double a, double b) {
    double r;
    __asm__("v_max_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// unsigned maximum over the wavefront, uniform
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false));  // row_shr:1
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false));  // row_shr:2
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false));  // row_shr:4
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false));  // row_shr:8
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));  // row_bcast:15
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));  // row_bcast:31
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// maximum of three keys as floats (NaN ignored)
__device__ __forceinline__ unsigned key_max3(unsigned a, unsigned b, unsigned c) {
    unsigned r;
    __asm__("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ unsigned hi_word(double v) {
    return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32);
}

// The pivot steps, by one wavefront.  S: 32 x 32 doubles (the symmetric copy), lbuf: the
// multipliers by row identity and pivot position.  On return bp holds the
// row at each position and the diagonal of S the uneliminated diagonal entries.
__device__ __forceinline__ int block_pivots(const double (*blk)[MAX_IB + 1], double *S, int *bp,
                                            int8_t *bkind, double *bdiag, double *boff, int bs, double small,
                                            double *maxl, double (*lbuf)[MAX_IB + 1]) {
    static_assert(MAX_IB == 32, "lane layout of the block");
    const int lane = fresh(threadIdx.x) & 63, i = lane & 31, h = lane >> 5;
    const double dead = __builtin_nan("");
    double e[8];
    int jo[8], w1[8], w2[8];  // column, and the entry's two places in S
    bool wild = false;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int j = (i + 1 + u + 8 * h) & 31;
        const bool copy2 = u == 7 && h == 1 && i >= 16;
        const double v = blk[max(i, j)][min(i, j)];
        const bool live = i < bs && j < bs;
        wild |= live && (hi_word(v) & 0x7fffffffu) >= 0x7e700000u;
        e[u] = (live && !copy2) ? v : dead;
        jo[u] = j;
        w1[u] = copy2 ? 33 * i : 32 * i + j;  // (the second copy writes its NaN to the diagonal)
        w2[u] = copy2 ? 33 * i : 32 * j + i;
    }
    double dg = blk[i][i];
    wild |= i < bs && (hi_word(dg) & 0x7fffffffu) >= 0x7e700000u;
    dg = (h == 0 && i < bs) ? dg : dead;
    if (h == 0) S[33 * i] = dead;
#pragma unroll
    for (int u = 0; u < 8; ++u) { S[w1[u]] = e[u]; S[w2[u]] = e[u]; }
    // a winning key above this is a value of at least `small` and far from the denormals
    const unsigned floor_key =
        __any(wild) ? 0xffffffffu : (unsigned)__builtin_amdgcn_readfirstlane((int)max(hi_word(small) | 31u, 0x01000000u));
    int posr = i, idr = i, pj[8];   // position of the lane's row and columns; row at position `lane`
#pragma unroll
    for (int u = 0; u < 8; ++u) pj[u] = jo[u];
    int kindr = 0;                  // lane c: kind and D of pivot c
    double bdr = 0.0, bor = 0.0;
    int cur = 0;
    double ml = 0.0;
    wave_sync();
    bool more = bs > 0;
    while (more) {
        unsigned long long mo, mg;
        unsigned M;
        // 1x1 pivots at the largest diagonal entry, clearly the largest entry of the block
        for (;;) {
            constexpr unsigned KEY = 0x7fffffe0u;
            unsigned ku[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) ku[u] = (hi_word(e[u]) & KEY) | (unsigned)jo[u];
            const unsigned kg = key_max3((hi_word(dg) & KEY) | (unsigned)i, 0u, 0u);
            const unsigned ko =
                key_max3(key_max3(ku[0], ku[1], ku[2]), key_max3(ku[3], ku[4], ku[5]), key_max3(ku[6], ku[7], 0u));
            M = wave_max_u32(max(kg, ko));
            // the row of the winner's column, which is the pivot's for a diagonal winner (the barrier
            // to the compiler keeps its loads here, in flight while the winner is checked)
            const int pid = M & 31;
            const double *row = S + 32 * pid;
            const double ci = row[i];
            double cj[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) cj[u] = row[jo[u]];
            __asm__ volatile("" ::: "memory");
            const unsigned T = M > floor_key ? M & ~31u : 0u;  // (0: every lane, so not this path)
            mo = __ballot(ko >= T);
            mg = __ballot(kg >= T);
            if ((mo | (mg & (mg - 1))) != 0) break;
            const double d = readlane_f64(dg, pid);
            const int pp = __builtin_amdgcn_readlane(posr, pid);
            const int x1 = __builtin_amdgcn_readlane(idr, cur);  // the row standing at position cur
            posr = (i == x1) ? pp : posr;
            idr = (lane == pp) ? x1 : idr;
            idr = (lane == cur) ? pid : idr;
            const double inv = 1.0 / d;
            const double li = ci * inv, wi = li * d;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                pj[u] = (jo[u] == x1) ? pp : pj[u];
                const double lj = cj[u] * inv, wj = lj * d;
                const double p1 = li * wj, p2 = lj * wi;
                e[u] = e[u] - (posr > pj[u] ? p1 : p2);
            }
            dg = dg - li * wi;
            ml = max_abs(ml, li);
            lbuf[i][cur] = li;
            kindr = (lane == cur) ? 1 : kindr;
            bdr = (lane == cur) ? d : bdr;
#pragma unroll
            for (int u = 0; u < 8; ++u) { S[w1[u]] = e[u]; S[w2[u]] = e[u]; }
            wave_sync();
            cur = __builtin_amdgcn_readfirstlane(cur + 1);
            if (cur >= bs) { more = false; break; }
        }
        if (!more) break;
        int ia, ib = M & 31;
        const unsigned long long mask = mo | mg;
        if (M > floor_key && (mask & (mask - 1)) == 0 && mg == 0) {
            ia = __builtin_ctzll(mask) & 31;
            // another entry of the winner's lane (all in row ia, or its diagonal) as large
            const double ca = S[32 * ia + i], g = fabs(readlane_f64(ca, ib));
            if ((__ballot(fabs(ca) >= g) & ~(0x100000001ull << ib)) != 0 || fabs(readlane_f64(dg, ia)) >= g) ia = -1;
        } else {
            ia = -1;
        }
        if (ia < 0) {
            // largest value, equal values by position; no live entry above zero: position cur
            const double m = max_abs(max_abs(max_abs(e[0], e[1]), max_abs(e[2], e[3])),
                                     max_abs(max_abs(e[4], e[5]), max_abs(e[6], e[7])));
            const double gv = wave_max_dpp(max_abs(max_abs(m, dg), 0.0));
            int key = (fabs(dg) == gv) ? 65 * posr : INT_MAX;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                key = (fabs(e[u]) == gv) ? min(key, 64 * min(posr, pj[u]) + max(posr, pj[u])) : key;
            key = (gv > 0.0) ? __builtin_amdgcn_readfirstlane(wave_min_int(key)) : 65 * cur;
            ia = __builtin_amdgcn_readlane(idr, key & 63);
            ib = __builtin_amdgcn_readlane(idr, key >> 6);
            if (gv < small) { more = false; break; }
        }
        // t: the winner's row (larger position), mi: its column
        const int qa = __builtin_amdgcn_readlane(posr, ia), qb = __builtin_amdgcn_readlane(posr, ib);
        const int t = qa > qb ? ia : ib, mi = qa > qb ? ib : ia;
        const double att = readlane_f64(dg, t), amm = readlane_f64(dg, mi);
        const double *r1 = S + 32 * mi, *r2 = S + 32 * t;
        const double a21 = r1[t];
        bool two = false;
        if (t != mi) {
            const double delta = amm * att - a21 * a21;
            two = fabs(delta) >= 0.5 * a21 * a21;
        }
        // the pivot's rows: a 2x2 takes mi to position cur, then t to cur + 1; a 1x1 the row with
        // the larger diagonal to cur
        const bool first = two || fabs(amm) >= fabs(att);
        auto move_to = [&](int pos, int id) {
            const int x = __builtin_amdgcn_readlane(idr, pos), q = __builtin_amdgcn_readlane(posr, id);
            posr = (i == x) ? q : (i == id) ? pos : posr;
            idr = (lane == q) ? x : idr;
            idr = (lane == pos) ? id : idr;
#pragma unroll
            for (int u = 0; u < 8; ++u) pj[u] = (jo[u] == x) ? q : (jo[u] == id) ? pos : pj[u];
        };
        move_to(cur, first ? mi : t);
        if (!two) {
            const double *rp = first ? r1 : r2;
            const double d = first ? amm : att;
            const double inv = 1.0 / d;
            const double li = rp[i] * inv, wi = li * d;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const double lj = rp[jo[u]] * inv, wj = lj * d;
                const double p1 = li * wj, p2 = lj * wi;
                e[u] = e[u] - (posr > pj[u] ? p1 : p2);
            }
            dg = dg - li * wi;
            ml = max_abs(ml, li);
            lbuf[i][cur] = li;
            kindr = (lane == cur) ? 1 : kindr;
            bdr = (lane == cur) ? d : bdr;
            cur += 1;
        } else {
            move_to(cur + 1, t);
            const double a11 = amm, a22 = att;
            const double inv_det = 1.0 / (a11 * a22 - a21 * a21);
            const double ci1 = r1[i], ci2 = r2[i];
            const double l1i = (ci1 * a22 - ci2 * a21) * inv_det;
            const double l2i = (ci2 * a11 - ci1 * a21) * inv_det;
            const double w1i = l1i * a11 + l2i * a21, w2i = l1i * a21 + l2i * a22;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const double cj1 = r1[jo[u]], cj2 = r2[jo[u]];
                const double l1j = (cj1 * a22 - cj2 * a21) * inv_det;
                const double l2j = (cj2 * a11 - cj1 * a21) * inv_det;
                const double w1j = l1j * a11 + l2j * a21, w2j = l1j * a21 + l2j * a22;
                const double p1 = l1i * w1j + l2i * w2j, p2 = l1j * w1i + l2j * w2i;
                e[u] = e[u] - (posr > pj[u] ? p1 : p2);
            }
            dg = dg - (l1i * w1i + l2i * w2i);
            ml = max_abs(max_abs(ml, l1i), l2i);
            lbuf[i][cur] = l1i;
            lbuf[i][cur + 1] = l2i;
            kindr = (lane == cur) ? 2 : (lane == cur + 1) ? 3 : kindr;
            bdr = (lane == cur) ? a11 : (lane == cur + 1) ? a22 : bdr;
            bor = (lane == cur) ? a21 : bor;
            cur += 2;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) { S[w1[u]] = e[u]; S[w2[u]] = e[u]; }
        wave_sync();
        cur = __builtin_amdgcn_readfirstlane(cur);
        more = cur < bs;
    }
    if (lane < MAX_IB) {
        bp[lane] = idr;
        S[33 * i] = dg;
        bkind[lane] = (int8_t)kindr;
        bdiag[lane] = bdr;
        boff[lane] = bor;
    }
    *maxl = wave_max_dpp(ml);
    return cur;
}

// All 256 threads: the block in blk (lower triangle) on entry; the factored block in position
// order on return (D's off-diagonal of a 2x2 at (q + 1, q)).  blk2, lbuf: working LDS.
// Wavefronts 1 to 3 call `beside` while the first runs the pivot steps.
template <class Beside>
__device__ __forceinline__ int block_factor_wg(double (*blk)[MAX_IB + 1], double (*blk2)[MAX_IB + 1], int *bp,
                                               int8_t *bkind, double *bdiag, double *boff, int bs, double small,
                                               double *maxl, double *wbv, int *wbp, double (*lbuf)[MAX_IB + 1],
                                               Beside beside) {
    const int tid = threadIdx.x;
    double *S = &blk2[0][0];
    if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) {
        __builtin_amdgcn_s_setprio(3);
        double ml;
        const int kk = block_pivots(blk, S, bp, bkind, bdiag, boff, bs, small, &ml, lbuf);
        __builtin_amdgcn_s_setprio(0);
        if (tid == 0) { wbv[0] = ml; wbp[0] = kk; }
    } else {
        beside();
    }
    lds_barrier();
    const int kk = __builtin_amdgcn_readfirstlane(wbp[0]);
    *maxl = wbv[0];
    // position (p, q): a multiplier of pivot q of the row now at p, D, or an uneliminated entry
    const int p = tid & (MAX_IB - 1);
    const int rid = bp[p];
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int q = (tid >> 5) + 8 * u;
        if (q > p || p >= bs) continue;
        double v;
        if (q >= kk) v = S[32 * rid + bp[q]];
        else if (p == q) v = bdiag[q];
        else v = (bkind[q] == 2 && p == q + 1) ? boff[q] : lbuf[rid][q];
        blk[p][q] = v;
    }
    lds_barrier();
    return kk;
}

// Substitution with L11 for a block that eliminated only bn < MAX_IB columns: columns and rows
// from bn on take no part.  Kept out of line: its guards are uniform predicates that, inlined,
// the compiler keeps live in registers across the common full-block path.
__device__ __attribute__((noinline)) void panel_trsm_partial(double *y, const double (*blk)[MAX_IB + 1], int bn) {
    const int lc = threadIdx.x & 31;
    double v[MAX_IB];
#pragma unroll
    for (int j = 0; j < MAX_IB; ++j) v[j] = y[j];
#pragma unroll
    for (int i = 0; i < MAX_IB - 1; ++i) {
        const double colv = blk[lc][i];
        if (i < bn) {
            const double yi = v[i];
#pragma unroll
            for (int j = i + 1; j < MAX_IB; ++j) {
                const double t = v[j] - readlane_f64(colv, j) * yi;
                v[j] = (j < bn) ? t : v[j];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < MAX_IB; ++j) y[j] = v[j];
}

// Forward substitution with a full L11 in groups: group (I, J) subtracts the terms of column I
// from rows J .. min(J + 8, MAX_IB) - 1; the groups run column by column, so every row receives
// its terms in ascending column order.  A group's eight products are formed before any of its
// subtractions (a scheduling barrier between them), so the products' latencies overlap instead
// of each subtraction waiting for its own product.
template <int I, int J>
struct TrsmNext {
    static constexpr bool more = J + 8 < MAX_IB;
    static constexpr int i = more ? I : I + 1;
    static constexpr int j = more ? J + 8 : I + 2;
    static constexpr bool valid = i < MAX_IB - 1;
};
template <int I, int J>
__device__ __forceinline__ void trsm_group_load(double (&c)[8], const double (*blk)[MAX_IB + 1]) {
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = (J + u < MAX_IB) ? blk[J + u < MAX_IB ? J + u : 0][I] : 0.0;
}
template <int I, int J>
__device__ __forceinline__ void trsm_groups(double (&y)[MAX_IB], const double (*blk)[MAX_IB + 1],
                                            const double (&c0)[8], const double (&c1)[8]) {
    using N1 = TrsmNext<I, J>;
    using N2 = TrsmNext<N1::i, N1::j>;
    double c2[8] = {};
    if constexpr (N1::valid && N2::valid) trsm_group_load<N2::i, N2::j>(c2, blk);
    const double yi = y[I];
    double t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (J + u < MAX_IB) t[u] = c0[u] * yi;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (J + u < MAX_IB) y[J + u] = y[J + u] - t[u];
    if constexpr (N1::valid) trsm_groups<N1::i, N1::j>(y, blk, c1, c2);
}

// Forward substitution with L11 and D^-1 for panel rows, one row per thread (factor.rs:1295-1408):
// y holds the row's block entries in pivot order on entry and its L entries on return.  blk is L11
// (2x2 D off-diagonals read as zeros), bkind / dinv / bdiag / boff the pivots (kind 0 beyond the
// eliminated columns).  L11's columns and the pivots' D sit in the lanes (lane c & 31 holds column
// / pivot c) and are taken by readlane: no LDS round trip per entry.  Every lane of the wavefront
// runs it (rows beyond the front hold zeros and store nothing), so the lanes read are active.
__device__ __forceinline__ void panel_trsm_d(double (&y)[MAX_IB], const double (*blk)[MAX_IB + 1], int bn,
                                             const int8_t *bkind, const double *dinv, const double *bdiag,
                                             const double *boff) {
    const int lc = threadIdx.x & 31;
    const int kdl = bkind[lc];
    const double dil = dinv[lc], bdl = bdiag[lc], bol = boff[lc];
    // forward substitution with L11 by columns: y[j] receives the terms of i = 0, 1, ...
    // in ascending order, as in the row form, while the rows stay independent
    if (bn == MAX_IB) {
        // every column eliminated (the common case): no guards, L11 entries read from LDS at
        // the same address by all lanes (broadcast), in groups of eight loaded two groups ahead
        double c0[8], c1[8];
        trsm_group_load<0, 1>(c0, blk);
        trsm_group_load<TrsmNext<0, 1>::i, TrsmNext<0, 1>::j>(c1, blk);
        trsm_groups<0, 1>(y, blk, c0, c1);
    } else {
        // through a copy: only the copy's address leaves the function, y stays in registers
        double t[MAX_IB];
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) t[j] = y[j];
        panel_trsm_partial(t, blk, bn);
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) y[j] = t[j];
    }
    // D^-1 (1x1: y / d; 2x2: Cramer's rule with the stored inverse determinant); columns beyond
    // the eliminated ones have kind 0 and stay as they are
#pragma unroll
    for (int c = 0; c < MAX_IB; ++c) {
        const int kd = __builtin_amdgcn_readlane(kdl, c);
        if (kd == 1) {
            y[c] *= readlane_f64(dil, c);
        } else if (kd == 2 && c + 1 < MAX_IB) {
            const double x1 = y[c], x2 = y[c + 1];
            const double di = readlane_f64(dil, c), bo = readlane_f64(bol, c);
            y[c] = (x1 * readlane_f64(bdl, c + 1) - x2 * bo) * di;
            y[c + 1] = (x2 * readlane_f64(bdl, c) - x1 * bo) * di;
        }
    }
}

// ===========================================================================
// APTP inner block, part 1 (one workgroup per 256 panel rows of a front): every workgroup
// factors the diagonal block itself (same arithmetic, same result), the first one records it --
// unless the previous update kernel already factored it (look-ahead, AptpState::pref); then each
// applies it to its panel rows -- backup, column permutation, TRSM with L11, D^-1 scaling and the
// a-posteriori threshold check (apply_and_check, factor.rs:1295-1408).
// ===========================================================================
__global__ __launch_bounds__(256) void k_block_apply(FrontDev *__restrict__ fr,
                                                     AptpState *__restrict__ st,
                                                     const int *__restrict__ flist,
                                                     const int4 *__restrict__ items, int ob,
                                                     int it, int nb, int ib, double small,
                                                     double threshold) {
    RV_PHASE_START();
    const int4 itm = items[blockIdx.x];
    const int li = itm.x, chunk = itm.y;
    FrontDev &F = fr[itm.z];
    AptpState &S = st[li];
    if (!aptp_active(F.k, nb, ib, ob, it)) return;
    const int k = S.kpos, m = F.m;
    const int bs = min(S.end_pos - k, ib), be = k + bs;
    const size_t lda = m;
    gdouble *A = gbl(F.F);
    // read once: a store through a front pointer may alias the state, so fields read after
    // stores would be reloaded before every one of them
    gdouble *const bk = gbl(S.backup);
    RV_PHASE_COUNT(0);
    RV_PHASE(0, 0);
    __shared__ double blk[MAX_IB][MAX_IB + 1];
    __shared__ int bp[MAX_IB], operm[MAX_IB];
    __shared__ int8_t bkind[MAX_IB];
    __shared__ double bdiag[MAX_IB], boff[MAX_IB], dinv[MAX_IB];
    __shared__ double wbv[1];
    __shared__ int wbp[1];
    __shared__ double lbuf[MAX_IB][MAX_IB + 1], blk2[MAX_IB][MAX_IB + 1];
    const int tid = threadIdx.x;
    const int r = be + chunk * 256 + tid;
    double y[MAX_IB];
    int bn;
    if (S.pref) {
        // the block was factored by the previous update kernel (look-ahead): its pivots, D and
        // L11 (2x2 D off-diagonals already zero) come from the state and the front; the panel
        // rows load directly in pivot order and are backed up in the original column order
        bn = S.block_nelim;
#ifdef RV_PHASE_TIMING
        if (blockIdx.x == 0 && tid == 0) atomicAdd(&g_phase[0][10], 1ull);
#endif
        if (tid < MAX_IB) {
            bp[tid] = S.bperm[tid];
            bkind[tid] = S.bkind[tid];
            bdiag[tid] = S.bdiag[tid];
            boff[tid] = S.boff[tid];
        }
        for (int e = tid; e < MAX_IB * MAX_IB; e += 256) {
            const int i = e & (MAX_IB - 1), j = e / MAX_IB;
            if (i < bs && j < i) blk[i][j] = A[(k + i) + (size_t)(k + j) * lda];
        }
        int pj[MAX_IB];
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) pj[j] = S.bperm[j];
        if (r < m) {
            gdouble *row = A + r;
#pragma unroll
            for (int j = 0; j < MAX_IB; ++j) y[j] = (j < bs) ? row[(size_t)(k + pj[j]) * lda] : 0.0;
#pragma unroll
            for (int j = 0; j < MAX_IB; ++j)
                if (j < bs) bk[(r - k) + (size_t)pj[j] * lda] = y[j];
        }
        lds_barrier();
        if (tid < bn) {
            const int kd = bkind[tid];
            if (kd == 1) dinv[tid] = 1.0 / bdiag[tid];
            else if (kd == 2) dinv[tid] = 1.0 / (bdiag[tid] * bdiag[tid + 1] - boff[tid] * boff[tid]);
        }
        lds_barrier();
        RV_PHASE(0, 3);
        if (bn == 0) return;
    } else {
    // every global load of the kernel's first part is issued before any is used: the panel
    // rows (backed up for restore_diagonal_with_perm), the lower block, the column order
    double pv[MAX_IB];
#pragma unroll
    for (int j = 0; j < MAX_IB; ++j) pv[j] = (r < m && j < bs) ? A[r + (size_t)(k + j) * lda] : 0.0;
    const int bi_ = tid & 31, bj0 = tid >> 5;
    double bv[MAX_IB / 8];
    const gdouble *const bc = gbl(S.blkcopy);
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int j = bj0 + 8 * u;
        const double v = bc[bi_ + j * MAX_IB];  // always in bounds (MAX_IB x MAX_IB)
        bv[u] = (bi_ < bs && j <= bi_) ? v : 0.0;
    }
    const int op = (chunk == 0 && tid < bs) ? gbl(F.perm)[k + tid] : 0;
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int j = bj0 + 8 * u;
        if (bi_ < bs && j <= bi_) {
            blk[bi_][j] = bv[u];
            if (chunk == 0) bk[bi_ + (size_t)j * lda] = bv[u];
        }
    }
    if (tid < MAX_IB) operm[tid] = op;
    lds_barrier();
    RV_PHASE(0, 1);
    double bml;
    bn = block_factor_wg(blk, blk2, bp, bkind, bdiag, boff, bs, small, &bml, wbv, wbp, lbuf, [] {});
    RV_PHASE(0, 2);
    // D off-diagonals of 2x2 pivots read as zeros of L11 (factor.rs:1898-1912)
    if (tid < bn) {
        const int kd = bkind[tid];
        if (kd == 2) blk[tid + 1][tid] = 0.0;
        if (kd == 1) dinv[tid] = 1.0 / bdiag[tid];
        else if (kd == 2) dinv[tid] = 1.0 / (bdiag[tid] * bdiag[tid + 1] - boff[tid] * boff[tid]);
    }
    if (r < m) {
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j)
            if (j < bs) bk[(r - k) + (size_t)j * lda] = pv[j];
    }
    lds_barrier();
    if (chunk == 0) {
        if (bn > 0) {
            const int i = tid & 31;
            for (int j = tid >> 5; j < bs; j += 8)
                if (i < bs && j <= i) A[(k + i) + (k + j) * lda] = blk[i][j];
            // column order by the block permutation (factor.rs:1926-1930)
            if (tid < bs) gbl(F.perm)[k + tid] = operm[bp[tid]];
        }
        if (tid < MAX_IB) {
            S.bperm[tid] = bp[tid];
            S.bkind[tid] = (tid < bn) ? bkind[tid] : 0;
            S.bdiag[tid] = bdiag[tid];
            S.boff[tid] = boff[tid];
        }
        if (tid == 0) {
            S.bs = bs;
            S.block_nelim = bn;
            atomicMin(&S.fail_min, bn);
            atomic_max_nonneg(&F.max_l_bits, bml);
        }
    }
    RV_PHASE(0, 3);
    if (bn == 0) return;
    if (r < m) {
        gdouble *row = A + r;
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) y[j] = (j < bs) ? row[(k + bp[j]) * lda] : 0.0;
    }
    }
    int first = INT_MAX;
    if (r >= m) {
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) y[j] = 0.0;
    }
    panel_trsm_d(y, blk, bn, bkind, dinv, bdiag, boff);
    if (r < m) {
        gdouble *row = A + r;
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j)
            if (j < bs) row[(k + j) * lda] = y[j];
        const double bound = 1.0 / threshold;
#pragma unroll
        for (int c = MAX_IB - 1; c >= 0; --c)
            if (c < bn && fabs(y[c]) >= bound) first = c;
        if (first != INT_MAX && bkind[first] == 3) first -= 1;
    }
    RV_PHASE(0, 4);
    // first failing column: wavefront minimum, one atomic per wavefront (no closing barrier)
    first = wave_min_int(first);
    if ((tid & 63) == 0 && first != INT_MAX) atomicMin(&S.fail_min, first);
    RV_PHASE(0, 5);
}

__device__ __forceinline__ double co_ld(const gdouble *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void co_st(gdouble *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int co_ldi(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void co_sti(int *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Bulk device-coherent loads: a plain buffer load carrying the same sc1 cache-policy bit as a
// device-scope atomic load, which the compiler batches like any other load (atomic loads are
// issued one round trip at a time).  The base is wavefront-uniform, the byte offset per lane; the
// resource's range turns an offset past it into zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t co_rsrc(const gdouble *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>((const double *)base), (short)0, 0x7FFFFFF0,
                                             0x00020000);
}
__device__ __forceinline__ double co_ldb(__amdgpu_buffer_rsrc_t r, size_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)(off * sizeof(double)), 0, 16));
}
// The same with the front's own end as the range (rows past a panel's last column would leave
// it); co_stb drops a store whose offset lies past the range.
constexpr unsigned CO_OOB = 0x7FFFFFF8u;  // (a column offset added to it stays past the range)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t co_rsrc_front(const gdouble *A, size_t lda, size_t off) {
    const size_t left = (lda * lda - off) * sizeof(double);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>((const double *)(A + off)), (short)0,
                                             (int)(left < 0x7FFFFFF0 ? left : 0x7FFFFFF0), 0x00020000);
}
__device__ __forceinline__ double co_ldo(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 16));
}
__device__ __forceinline__ void co_stb(__amdgpu_buffer_rsrc_t r, unsigned off, double v) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, (int)off, 0, 16);
}
__device__ __forceinline__ void co_std(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// every thread's stores complete, then the workgroup barrier
__device__ __forceinline__ void stores_done_barrier() {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// ===========================================================================
// Symmetric line permutation for a sequence of at most MAX_IB swap_symmetric calls (factor.rs:452-505):
// the composite touches at most 2 MAX_IB lines U.  Outside U x U every other line q is independent:
// a thread loads its q's entries of up to RL touched lines (whole cycles of the permutation, all
// loads of a round in flight) and stores them to the lines' new places; the U x U entries go
// through S.swapbuf.  RL: MAX_IB, or half of that where a launch of thousands of workgroups, most of them
// without a swap, should hold eight wavefronts per SIMD (k_block_finish).  CO: device-scope accesses to the front (inside the persistent launch, where
// the panels share the other lines).
// apply_swaps is out of line: its registers stay out of the callers' common path.  Snapshotting whole lines to
// memory one element and round trip at a time took a quarter of the factorization of a KKT system
// with many delays (side 45: 28.4 ms, 21.9 so); by the leader of the persistent launch alone the
// lines still took 88 us a block, shared between its workgroups the step went from 17.9 to 13.6 ms.
// ===========================================================================
struct SwapLds {
    int U[2 * MAX_IB];     // touched lines
    int from[2 * MAX_IB];  // line i receives line from[i] (indices into U)
    int ptmp[2 * MAX_IB];
    int mv[2 * MAX_IB];    // moved lines cycle by cycle: destination index, + 64 where a cycle ends
    int gend[2 * MAX_IB];  // rounds of at most RL moves (whole cycles): end in mv
    int n, nmv, ng;        // (ng = 0: a cycle of more than RL lines)
};
// The plan of a sequence of nsw swaps (all threads; ends with the barrier).
template <int RL>
__device__ __forceinline__ void swap_plan(SwapLds &W, const int *sa, const int *sb, int nsw) {
    static_assert(MAX_IB == 32, "a touched line per lane");
    const int lane = threadIdx.x & 63;
    if (threadIdx.x < 64) {
        // lane i: touched line i and the line whose content it ends with
        int line = -1, from = lane, nU = 0;
        const int la = lane < nsw ? sa[lane] : 0, lb = lane < nsw ? sb[lane] : 0;
        for (int s = 0; s < nsw; ++s) {
            const int x = __builtin_amdgcn_readlane(la, s), y = __builtin_amdgcn_readlane(lb, s);
            auto find = [&](int v) {
                const unsigned long long hit = __ballot(lane < nU && line == v);
                if (hit) return (int)__builtin_ctzll(hit);
                line = (lane == nU) ? v : line;
                return nU++;
            };
            const int ix = find(x), iy = find(y);
            const int fx = __builtin_amdgcn_readlane(from, ix), fy = __builtin_amdgcn_readlane(from, iy);
            from = (lane == ix) ? fy : (lane == iy) ? fx : from;
        }
        W.U[lane] = line;
        W.from[lane] = from;
        // the cycles, dealt to rounds
        unsigned long long left = __ballot(from != lane);
        int k = 0, g0 = 0, ng = 0;
        bool longc = false;
        while (left) {
            const int first = __builtin_ctzll(left), k0 = k;
            int c = first;
            do {
                left &= ~(1ull << c);
                const int nx = __builtin_amdgcn_readlane(from, c);
                if (lane == 0) W.mv[k] = c + (nx == first ? 64 : 0);
                ++k;
                c = nx;
            } while (c != first);
            longc |= k - k0 > RL;
            if (k - g0 > RL) {
                if (lane == 0) W.gend[ng] = k0;
                ++ng;
                g0 = k0;
            }
        }
        if (lane == 0) {
            W.gend[ng] = k;
            W.n = nU;
            W.nmv = k;
            W.ng = longc ? 0 : ng + 1;
        }
    }
    __syncthreads();
}

// The touched lines' crossings with the lines [q_begin, q_end) outside U; a wavefront takes 64 of
// these and one round.
template <bool CO, int RL>
__device__ __forceinline__ void swap_lines(FrontDev &F, const SwapLds &W, int q_begin, int q_end) {
    constexpr int AUX = CO ? 16 : 0;
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = F.m;
    const size_t lda = m;
    gdouble *A = gbl(F.F);
    const int nU = __builtin_amdgcn_readfirstlane(W.n), nmv = __builtin_amdgcn_readfirstlane(W.nmv);
    const bool near = (size_t)m * m < (1u << 27);  // the front's offsets fit a buffer resource
    const __amdgpu_buffer_rsrc_t ra = co_rsrc(A);
    const int ul = W.U[lane], fl = W.from[lane], ml = W.mv[lane] & 63;
    const int ng = near ? __builtin_amdgcn_readfirstlane(W.ng) : 0, ngx = max(ng, 1);
    const int ntask = (q_end - q_begin + 63) / 64 * ngx;
    // (every lane stays active: the lines are read across the lanes)
    for (int task = wv; task < ntask; task += nw) {
        const int g = task % ngx, q = q_begin + task / ngx * 64 + lane;
        bool in = q < q_end;
        for (int s = 0; s < nU; ++s) in = in && q != __builtin_amdgcn_readlane(ul, s);
        if (ng > 0) {
            const int g0 = g > 0 ? __builtin_amdgcn_readfirstlane(W.gend[g > 0 ? g - 1 : 0]) : 0;
            const int n = __builtin_amdgcn_readfirstlane(W.gend[g]) - g0;
            double v[RL];
#pragma unroll
            for (int s = 0; s < RL; ++s)
                if (s < n) {
                    const int u = __builtin_amdgcn_readlane(ul, __builtin_amdgcn_readlane(fl, __builtin_amdgcn_readlane(ml, g0 + s)));
                    const unsigned off = in ? 8u * ((unsigned)max(q, u) + (unsigned)min(q, u) * (unsigned)m) : CO_OOB;
                    v[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ra, (int)off, 0, AUX));
                }
#pragma unroll
            for (int s = 0; s < RL; ++s)
                if (s < n) {
                    const int u = __builtin_amdgcn_readlane(ul, __builtin_amdgcn_readlane(ml, g0 + s));
                    const unsigned off = in ? 8u * ((unsigned)max(q, u) + (unsigned)min(q, u) * (unsigned)m) : CO_OOB;
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v[s]), ra, (int)off, 0, AUX);
                }
        } else if (in) {
            // a long cycle, or a front of 1 GiB (order 11586) or more: along each cycle, the first entry kept aside
            double first = 0.0;
            bool start = true;
            for (int s = 0; s < nmv; ++s) {
                const int w = W.mv[s], i = w & 63, u = W.U[i], f = W.U[W.from[i]];
                gdouble *pu = A + max(q, u) + (size_t)min(q, u) * lda, *pf = A + max(q, f) + (size_t)min(q, f) * lda;
                if (start) first = CO ? co_ld(pu) : *pu;
                const double x = (w & 64) ? first : CO ? co_ld(pf) : *pf;
                if (CO) co_st(pu, x);
                else *pu = x;
                start = (w & 64) != 0;
            }
        }
    }
}

// The touched lines' crossings with each other (through S.swapbuf) and the row order.
template <bool CO>
__device__ __forceinline__ void swap_cross(FrontDev &F, AptpState &S, SwapLds &W) {
    constexpr int AUX = CO ? 16 : 0;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int m = F.m;
    const size_t lda = m;
    gdouble *A = gbl(F.F);
    const int nU = __builtin_amdgcn_readfirstlane(W.n);
    gdouble *buf = gbl(S.swapbuf);
    const bool near = (size_t)m * m < (1u << 27);  // the front's offsets fit a buffer resource
    const __amdgpu_buffer_rsrc_t ra = co_rsrc(A);
    for (int e0 = tid; e0 < nU * nU; e0 += nt * 8) {
        double v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int e = e0 + nt * r, x = e < nU * nU ? e / nU : 0, y = e < nU * nU ? e % nU : 0;
            const size_t off = W.U[x] + (size_t)W.U[y] * lda;
            const bool ok = e < nU * nU && W.U[x] >= W.U[y];
            if (near)
                v[r] = __builtin_bit_cast(
                    double, __builtin_amdgcn_raw_buffer_load_b64(ra, (int)(ok ? (unsigned)off * 8u : CO_OOB), 0, AUX));
            else
                v[r] = ok ? co_ld(A + off) : 0.0;
        }
#pragma unroll
        for (int r = 0; r < 8; ++r)
            if (e0 + nt * r < nU * nU) buf[e0 + nt * r] = v[r];
    }
    if (tid < nU) W.ptmp[tid] = gbl(F.perm)[W.U[tid]];
    __syncthreads();
    for (int e = tid; e < nU * nU; e += nt) {
        const int x = e / nU, y = e % nU;
        const int p = W.U[x], r = W.U[y];
        if (p < r) continue;
        const int fx = W.from[x], fy = W.from[y];
        const double v = buf[W.U[fx] >= W.U[fy] ? fx * nU + fy : fy * nU + fx];
        if (CO) co_st(A + p + (size_t)r * lda, v);
        else A[p + (size_t)r * lda] = v;
    }
    if (tid < nU) gbl(F.perm)[W.U[tid]] = W.ptmp[W.from[tid]];
}

// The whole permutation by one workgroup.
template <int RL>
__device__ __forceinline__ void apply_swaps_inline(FrontDev &F, AptpState &S, const int *sa, const int *sb, int nsw,
                                                   SwapLds &W) {
    swap_plan<RL>(W, sa, sb, nsw);
    if (W.nmv > 0) {
        swap_cross<false>(F, S, W);
        swap_lines<false, RL>(F, W, 0, F.m);
    }
    __syncthreads();
}

__device__ __attribute__((noinline)) void apply_swaps(FrontDev &F, AptpState &S, const int *sa, const int *sb, int nsw,
                                                      SwapLds &W) {
    apply_swaps_inline<MAX_IB>(F, S, sa, sb, nsw, W);
}

// Inside the persistent launch the permutation is shared: the leader's part (part < 0), and part of
// np of the other lines.  Ends with the workgroup's stores complete.
__device__ __forceinline__ void apply_swaps_shared(FrontDev &F, AptpState &S, const int *sa, const int *sb,
                                                             int nsw, SwapLds &W, int part, int np) {
    swap_plan<MAX_IB>(W, sa, sb, nsw);
    if (W.nmv > 0) {
        if (part < 0) {
            swap_cross<true>(F, S, W);
        } else {
            const int per = (F.m + np - 1) / np;
            swap_lines<true, MAX_IB>(F, W, min(part * per, F.m), min((part + 1) * per, F.m));
        }
    }
    stores_done_barrier();
}

// The swaps that move block [k, k + bs)'s failed columns (from nelim on; all with bn == 0) to the end
// of the outer block: one thread; returns their number, end_pos is moved.
__device__ __forceinline__ int failed_swaps(int k, int bs, int bn, int nelim, int &end_pos, int *sa, int *sb) {
    int n = 0;
    if (bn == 0) {
        for (int off = 0; off < bs; ++off) {
            end_pos -= 1;
            if (k + off < end_pos) { sa[n] = k + off; sb[n] = end_pos; ++n; }
        }
    } else {
        for (int i = bs - nelim - 1; i >= 0; --i) {
            const int dp = k + nelim + i;
            end_pos -= 1;
            if (dp < end_pos) { sa[n] = dp; sb[n] = end_pos; ++n; }
        }
    }
    return n;
}

// Diagonal tile of the next inner block after this block's update, formed in LDS with the
// trailing update's arithmetic: C(i, c) -= sum_j W(i, j) L(c, j), summed over j ascending from
// zero and subtracted once.  Lr holds the next block's L rows in this block's columns, kd / dd /
// od this block's pivots; Wt receives W = L D (compute_ld_into, factor.rs:1536-1563).  Thread
// (ii = tid & 31, jg = tid >> 5) returns its updated entries (ii, jg + 8u) in nv.  Starts with the
// LDS operands in place and ends with a barrier.
__device__ __forceinline__ void next_tile_update(const double (*Lr)[MAX_IB + 1], double (*Wt)[MAX_IB + 1],
                                                 double (*Ct)[MAX_IB + 1], const int8_t *kd, const double *dd,
                                                 const double *od, int nbs, int nelim,
                                                 double (&nv)[MAX_IB / 8]) {
    const int tid = threadIdx.x, ii = tid & 31, jg = tid >> 5;
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int j = jg + 8 * u;
        double w = 0.0;
        if (ii < nbs && j < nelim) {
            const int kj = kd[j];
            if (kj == 1) w = Lr[ii][j] * dd[j];
            else if (kj == 2) w = Lr[ii][j] * dd[j] + Lr[ii][j + 1] * od[j];
            else if (kj == 3) w = Lr[ii][j - 1] * od[j - 1] + Lr[ii][j] * dd[j];
        }
        Wt[ii][j] = w;
    }
    lds_barrier();
    // the thread's four sums run side by side (independent chains, one W read per step); a full
    // block without guards, so the LDS reads of later steps are issued ahead
    double sacc[MAX_IB / 8];
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) sacc[u] = 0.0;
    if (nelim == MAX_IB) {
        // operands of step j + 2 loaded during step j (three register sets in turn), a scheduling
        // barrier per step so that the loads are not regrouped behind their uses
        double wq[3], lq[3][MAX_IB / 8];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            wq[j] = Wt[ii][j];
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) lq[j][u] = Lr[jg + 8 * u][j];
        }
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) {
            if (j + 2 < MAX_IB) {
                wq[(j + 2) % 3] = Wt[ii][j + 2];
#pragma unroll
                for (int u = 0; u < MAX_IB / 8; ++u) lq[(j + 2) % 3][u] = Lr[jg + 8 * u][j + 2];
            }
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) sacc[u] += wq[j % 3] * lq[j % 3][u];
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int j = 0; j < MAX_IB; ++j) {
            if (j < nelim) {
                const double w = Wt[ii][j];
#pragma unroll
                for (int u = 0; u < MAX_IB / 8; ++u) sacc[u] += w * Lr[jg + 8 * u][j];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int c = jg + 8 * u;
        nv[u] = 0.0;
        if (ii < nbs && c <= ii) {
            nv[u] = Ct[ii][c] - sacc[u];
            Ct[ii][c] = nv[u];
        }
    }
    lds_barrier();
}

// Look-ahead factorization of the next inner block [be, be + nbs), by one extra workgroup per
// front of the update kernel.  It forms the block's diagonal tile after this block's update on its
// own -- C - sum_j w_j l_j over the block's eliminated columns in ascending order (the arithmetic
// of the trailing update, which writes the same tile to the front), with every operand loaded in
// one round trip -- and then takes the steps of k_block_apply's staging part: backup of the block,
// complete pivoting, D off-diagonals of 2x2 pivots zeroed in L11, the factored block and the
// column order written to the front; pivots and D go to the nx_* fields, which k_block_finish
// hands over.  Wr (64 x 33) and Lc (32 x 33) are its LDS.
constexpr int LOOKAHEAD_Q = 255;  // k_block_update work item of the look-ahead workgroup

__device__ void lookahead_factor(FrontDev &F, AptpState &S, double (*Wr)[MAX_IB + 1], double (*Lc)[MAX_IB + 1],
                                 int k, int be, int nelim, int nbs, double small, unsigned long long t_start) {
    // the chain below is the critical path of the update kernel: its wavefronts issue first
    __builtin_amdgcn_s_setprio(3);
#ifdef RV_PHASE_TIMING
    const bool probe = threadIdx.x == 0 && blockIdx.x < 64;
    if (probe) { atomicAdd(&g_phase[1][6], clock64() - t_start); atomicAdd(&g_phase[1][5], 1ull); }
    const unsigned long long t0 = clock64();
#endif
    __shared__ int bp[MAX_IB], operm[MAX_IB];
    __shared__ int8_t bkind[MAX_IB];
    __shared__ double bdiag[MAX_IB], boff[MAX_IB];
    __shared__ double wbv[1];
    __shared__ int wbp[1];
    __shared__ int8_t kd[MAX_IB];
    __shared__ double dd[MAX_IB], od[MAX_IB];
    double (*Lr)[MAX_IB + 1] = Wr;            // L rows of the next block in this block's columns
    double (*Wt)[MAX_IB + 1] = Wr + MAX_IB;   // their W = L D
    double (*Ct)[MAX_IB + 1] = Lc;            // the diagonal tile, updated in place
    const int tid = threadIdx.x;
    const size_t lda = F.m;
    gdouble *A = gbl(F.F);
    gdouble *const bk = gbl(S.backup);
    // one round trip: D of this block, the L rows, the tile, the column order
    const int ii = tid & 31, jg = tid >> 5;
    double lv[MAX_IB / 8], cv[MAX_IB / 8];
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int j = jg + 8 * u;
        lv[u] = (ii < nbs && j < nelim) ? A[(be + ii) + (size_t)(k + j) * lda] : 0.0;
        cv[u] = (ii < nbs && j <= ii) ? A[(be + ii) + (size_t)(be + j) * lda] : 0.0;
    }
    int8_t kv = 0;
    double dv = 0.0, ov = 0.0;
    int opv = 0;
    if (tid < MAX_IB) {
        kv = S.bkind[tid];
        dv = S.bdiag[tid];
        ov = S.boff[tid];
        opv = (tid < nbs) ? gbl(F.perm)[be + tid] : 0;
    }
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int j = jg + 8 * u;
        Lr[ii][j] = lv[u];
        Ct[ii][j] = cv[u];
    }
    if (tid < MAX_IB) { kd[tid] = kv; dd[tid] = dv; od[tid] = ov; operm[tid] = opv; }
    lds_barrier();
    double nv[MAX_IB / 8];
    next_tile_update(Lr, Wt, Ct, kd, dd, od, nbs, nelim, nv);
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int c = jg + 8 * u;
        if (ii < nbs && c <= ii) bk[ii + (size_t)c * lda] = nv[u];
    }
    double bml;
#ifdef RV_PHASE_TIMING
    if (probe) atomicAdd(&g_phase[1][2], clock64() - t0);
#endif
    const int bn = block_factor_wg(Ct, Wr, bp, bkind, bdiag, boff, nbs, small, &bml, wbv, wbp, Wr + MAX_IB,
                                   [] {});
#ifdef RV_PHASE_TIMING
    if (probe) atomicAdd(&g_phase[1][3], clock64() - t0);
#endif
    double (*blk)[MAX_IB + 1] = Ct;
    if (tid < bn && bkind[tid] == 2) blk[tid + 1][tid] = 0.0;
    lds_barrier();
    // the tile goes back to the front also when nothing was eliminated: the update kernel leaves
    // it to this workgroup, so the front holds it only from here
    {
        const int i2 = tid & 31;
        for (int j = tid >> 5; j < nbs; j += 8)
            if (i2 < nbs && j <= i2) A[(be + i2) + (size_t)(be + j) * lda] = blk[i2][j];
    }
    if (bn > 0 && tid < nbs) gbl(F.perm)[be + tid] = operm[bp[tid]];
    if (tid < MAX_IB) {
        S.nx_bperm[tid] = bp[tid];
        S.nx_bkind[tid] = (tid < bn) ? bkind[tid] : 0;
        S.nx_bdiag[tid] = bdiag[tid];
        S.nx_boff[tid] = boff[tid];
    }
    if (tid == 0) {
        S.nx_bs = nbs;
        S.nx_bn = bn;
        S.nx_valid = 1;
        atomic_max_nonneg(&F.max_l_bits, bml);
    }
#ifdef RV_PHASE_TIMING
    if (probe) atomicAdd(&g_phase[1][4], clock64() - t0);
#endif
    __builtin_amdgcn_s_setprio(0);
}

// ===========================================================================
// APTP inner block, part 2 (tiles of 64 rows x 32 columns relative to kpos; column tile 0 =
// the current block): partial restore of failed columns, cross terms, Schur update of the
// trailing columns of the outer block, max|L| statistics (factor.rs:1945-2008:
// restore_diagonal_with_perm, update_trailing, update_cross_terms), and the block row
// permutation of the already-factored columns (factor.rs:1914-1924).
// ===========================================================================
__global__ __launch_bounds__(256) void k_block_update(FrontDev *__restrict__ fr,
                                                      AptpState *__restrict__ st,
                                                      const int *__restrict__ flist,
                                                      const int4 *__restrict__ items, int ob,
                                                      int it, int nb, int ib, double small) {
    RV_PHASE_START();
    RV_PHASE_COUNT(1);
    const int4 itm = items[blockIdx.x];
    const int li = itm.x, rt = itm.y, q = itm.z;
    FrontDev &F = fr[itm.w];
    AptpState &S = st[li];
    if (!aptp_active(F.k, nb, ib, ob, it)) return;
    const int bn = S.block_nelim;
    const int k = S.kpos, bs = S.bs, be = k + bs, m = F.m;
    // trailing columns updated by this inner block: every fully-summed column, as
    // update_trailing does (factor.rs:1418-1526 with nfs_boundary, 2149), or only those of the
    // current outer block when the rest is deferred to the rank-nb MFMA update
    const int obe = (F.flags & FRONT_ALLFS) ? F.k : S.ob_start + S.ob_cols;
    const size_t lda = m;
    gdouble *A = gbl(F.F);
    gdouble *const bk = gbl(S.backup);
    const int nelim = (bn > 0) ? effective_nelim(S) : 0;
    __shared__ double Wr[64][MAX_IB + 1];
    __shared__ double Lc[32][MAX_IB + 1];
    __shared__ int bp[MAX_IB];
    __shared__ int kind[MAX_IB];
    __shared__ double dg[MAX_IB], of[MAX_IB];
    const int tid = threadIdx.x;
    // look-ahead: after a block without failures, the next block [be, be + nbs) is factored by an
    // extra workgroup (only when the next inner-block launch will process it: the look-ahead
    // writes it); its diagonal tile is then that workgroup's alone
    const int nbs = min(S.end_pos - be, ib);
    const bool ahead = bn > 0 && nelim == bs && nbs > 0 && aptp_active(F.k, nb, ib, ob, it + 1);
    if (q == LOOKAHEAD_Q) {
        if (ahead) {
#ifdef RV_PHASE_TIMING
            const unsigned long long t_start = rv_t0_;
#else
            const unsigned long long t_start = 0;
#endif
            lookahead_factor(F, S, Wr, Lc, k, be, nelim, nbs, small, t_start);
        }
        return;
    }
    RV_PHASE(1, 0);
    if (tid < MAX_IB) {
        bp[tid] = S.bperm[tid];
        kind[tid] = S.bkind[tid];
        dg[tid] = S.bdiag[tid];
        of[tid] = S.boff[tid];
    }
    lds_barrier();
    int c_lo, c_hi;
    bool active = bn > 0;
    if (q == 0) { c_lo = k; c_hi = be; }
    else {
        c_lo = be + 32 * (q - 1);
        c_hi = min(c_lo + 32, obe);
        if (c_lo >= obe || nelim == 0) active = false;
    }
    const int r_lo = k + 64 * rt;
    const int r_hi = min(r_lo + 64, m);
    if (r_lo >= m || (q >= 1 && r_hi <= c_lo)) active = false;
    if (active) {
        const int ncol = c_hi - c_lo;
        for (int e = tid; e < 64 * nelim; e += 256) {
            const int rr = e & 63, j = e >> 6;
            const int r = r_lo + rr;
            Wr[rr][j] = (r < r_hi) ? ld_entry(A + r + k * lda, lda, j, kind[j], dg, of) : 0.0;
        }
        if (q >= 1) {
            for (int e = tid; e < 32 * nelim; e += 256) {
                const int cc = e & 31, j = e >> 5;
                if (cc < ncol) Lc[cc][j] = A[(c_lo + cc) + (k + j) * lda];
            }
        } else {
            // L rows of the failed block rows: Lc[jf][c] = A(k+nelim+jf, k+c)
            const int nf = bs - nelim;
            for (int e = tid; e < 32 * nelim; e += 256) {
                const int jf = e & 31, c = e >> 5;
                if (jf < nf) Lc[jf][c] = A[(k + nelim + jf) + (k + c) * lda];
            }
        }
        lds_barrier();
        const int rr = tid & 63;
        const int r = r_lo + rr;
        const bool valid = r < r_hi;
        gdouble *row = A + r;
        if (q >= 1) {
            if (valid) {
                // the row's W values stay in registers across the tile's columns; each sum runs
                // over c ascending from zero and is subtracted once (gemm_sub_wlt order)
                double w[MAX_IB];
#pragma unroll
                for (int j = 0; j < MAX_IB; ++j) w[j] = Wr[rr][j];
                // the row's 8 entries are loaded before any is stored (a store may alias a later
                // load, so interleaved read-modify-writes would take one round trip each)
                double cv[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int cc = (tid >> 6) + 4 * u;
                    const int c = c_lo + cc;
                    const bool tile_ahead = ahead && r < be + nbs && c < be + nbs;
                    cv[u] = (cc < ncol && r >= c && !tile_ahead) ? row[c * lda] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int cc = (tid >> 6) + 4 * u;
                    const int c = c_lo + cc;
                    const bool tile_ahead = ahead && r < be + nbs && c < be + nbs;
                    if (cc < ncol && r >= c && !tile_ahead) {
                        double s = 0.0;
#pragma unroll
                        for (int j = 0; j < MAX_IB; ++j)
                            if (j < nelim) s += w[j] * Lc[cc][j];
                        row[c * lda] = cv[u] - s;
                    }
                }
            }
        } else {
            double ml = 0.0;
            for (int j = tid >> 6; valid && j < bs; j += 4) {
                const int c = k + j;
                if (j >= nelim) {
                    // partial restore (only when the check removed pivots)
                    if (nelim < bn) {
                        if (r < be) {
                            const int i = r - k;
                            if (i >= j) {
                                const int br = bp[i], bc = bp[j];
                                row[c * lda] = (br >= bc) ? bk[br + bc * lda] : bk[bc + br * lda];
                            }
                        } else {
                            row[c * lda] = bk[(r - k) + bp[j] * lda];
                        }
                    }
                    // cross terms from the passed columns
                    if (nelim > 0) {
                        const int jf = j - nelim;
                        const bool below = r >= be;
                        if (below || r - k - nelim >= jf) {
                            double s = 0.0;
                            for (int cc2 = 0; cc2 < nelim; ++cc2) s += Wr[rr][cc2] * Lc[jf][cc2];
                            row[c * lda] -= s;
                        }
                    }
                } else if (r >= be) {
                    const double v = fabs(row[c * lda]);
                    if (v > ml) ml = v;
                }
            }
            ml = wave_fmax(ml);
            if ((tid & 63) == 0) atomic_max_nonneg(&F.max_l_bits, ml);
        }
    }
    if (q == 0 && bn > 0) {
        // block rows permuted in the columns factored before this block: two columns per
        // wavefront instruction, lane&31 = row of the block
        const int ntr = (m + 63) / 64;
        const int per = (k + ntr - 1) / ntr;
        const int cb = rt * per, ce = min(k, cb + per);
        const int i = tid & 31, half = (tid >> 5) & 1, wv = tid >> 6;
        if (i < bs) {
            const int src = k + bp[i];
            for (int c0 = cb + 2 * wv + half; c0 < ce; c0 += 32) {
                double v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int c = c0 + 8 * u;
                    v[u] = (c < ce) ? A[src + (size_t)c * lda] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int c = c0 + 8 * u;
                    if (c < ce) A[(k + i) + (size_t)c * lda] = v[u];
                }
            }
        }
    }
    RV_PHASE(1, 1);
}

// End of an inner block (one workgroup per front): D and the pivot counts of the accepted
// columns, then the failed columns are delayed to the end of the outer block
// (factor.rs:1962-2077).
__global__ __launch_bounds__(256) void k_block_finish(FrontDev *__restrict__ fr,
                                                      AptpState *__restrict__ st,
                                                      const int *__restrict__ flist, int ob, int it,
                                                      int nb, int ib) {
    const int li = blockIdx.x;
    FrontDev &F = fr[flist[li]];
    AptpState &S = st[li];
    if (!aptp_active(F.k, nb, ib, ob, it)) return;
    const int tid = threadIdx.x;
    const int bn = S.block_nelim;
    const int k = S.kpos, bs = S.bs;
    const int nelim = (bn > 0) ? effective_nelim(S) : 0;
    const int nxv = S.nx_valid;
    __shared__ int sa[MAX_IB], sb[MAX_IB];
    __shared__ SwapLds sw;
    __shared__ int nsw, s_end;
    int is1 = 0, is2 = 0;
    if (tid < nelim) {
        const int kd = S.bkind[tid];
        const int c = k + tid;
        if (kd == 1) {
            gbl(F.dkind)[c] = 1; gbl(F.ddiag)[c] = S.bdiag[tid]; gbl(F.doff)[c] = 0.0;
            is1 = 1;
        } else if (kd == 2 && tid + 1 < nelim) {
            gbl(F.dkind)[c] = 2; gbl(F.dkind)[c + 1] = 3;
            gbl(F.ddiag)[c] = S.bdiag[tid]; gbl(F.ddiag)[c + 1] = S.bdiag[tid + 1];
            gbl(F.doff)[c] = S.boff[tid]; gbl(F.doff)[c + 1] = 0.0;
            is2 = 1;
        }
    }
    const int n1 = __syncthreads_count(is1);
    const int n2 = __syncthreads_count(is2);
    if (tid == 0) {
        F.n1 += n1;
        F.n2 += n2;
        int end_pos = S.end_pos;
        nsw = failed_swaps(k, bs, bn, nelim, end_pos, sa, sb);
        s_end = end_pos;
    }
    __syncthreads();
    // (with the swaps of RL = MAX_IB out of line the launch took 196 registers: 50 us for 4000 fronts
    // without a failed column, 16 so)
    if (nsw > 0) apply_swaps_inline<MAX_IB / 2>(F, S, sa, sb, nsw, sw);
    if (tid == 0) {
        S.kpos = k + nelim;
        S.end_pos = s_end;
        S.fail_min = INT_MAX;
        if (S.nib < MAX_OB_IB) S.ib_ne[S.nib] = (int8_t)nelim;
        S.nib += 1;
    }
    __syncthreads();
    if (nxv) {
        // the next block was factored ahead by the update kernel (this block had no failures,
        // so nothing moved): its pivots and D become the current block's
        if (tid < MAX_IB) {
            S.bperm[tid] = S.nx_bperm[tid];
            S.bkind[tid] = S.nx_bkind[tid];
            S.bdiag[tid] = S.nx_bdiag[tid];
            S.boff[tid] = S.nx_boff[tid];
        }
        if (tid == 0) {
            S.bs = S.nx_bs;
            S.block_nelim = S.nx_bn;
            S.fail_min = S.nx_bn;
            S.pref = 1;
            S.nx_valid = 0;
        }
    } else {
        if (tid == 0) S.pref = 0;
        if (S.kpos < S.end_pos) copy_next_block(F, S, ib);
    }
}

// ===========================================================================
// APTP outer block in one persistent launch (k_aptp_outer), for levels whose workgroups all fit
// on the device at once.  Per front one leader workgroup runs the pivot chain and NP panel
// workgroups own chunks of CH rows from the outer block's first column down:
//   leader, inner block it: factor the diagonal block (or take the one factored ahead), publish
//     its pivots and L11 (record it); then, when the block eliminated every column, form the next
//     block's L rows itself (the panel substitution for those 32 rows), its diagonal tile after
//     this block's update, factor that tile ahead and write its record, unpublished; meanwhile two
//     of its wavefronts store the current tile (they count among the NP + 2 of `applied`), and
//     while one runs the pivots the others bring the operands of the block after it once the
//     panels that own them report (`early`).  When every panel has checked block it, the next
//     record is published if no column failed; after failures the panels' restores are awaited,
//     the failed columns move to the end of the outer block (the panels swap the lines, `swapped`)
//     and the next block is factored afresh.
//   panel, inner block it: backup, column permutation, substitution and threshold check of its
//     rows (k_block_apply), then, once every panel has checked, partial restore and cross terms,
//     the update of the outer block's trailing columns in its rows (the tile factored ahead left
//     to the leader) and its share of the row permutation of earlier columns (k_block_update).
// The arithmetic of every entry is the three-kernel path's, so both produce the same bits.
// Front entries, backups and records that one workgroup writes and another reads within the
// launch go through device-scope loads and stores, which bypass the per-XCD L2 (another XCD's
// copy would be stale); a producer's stores complete (s_waitcnt) before it bumps a counter, and a
// consumer's thread 0 spins on the counter with device-scope loads (bounded: a wait that runs out
// sets the front's error word, every wait of the front then gives up, and the host discards the
// launch's results).
// ===========================================================================
constexpr int CHAIN_MAX_IT = 8;                 // inner blocks per outer block
constexpr long long CHAIN_SPIN_LIMIT = 1ll << 22;
constexpr int FRONT_CHAIN_ERR = 8;              // FrontDev::flags: a wait of k_aptp_outer ran out
constexpr int FRONT_LA_ERR = 16;   // FrontDev::flags: an outer block run with its trailing update
                                   // overlapped (no failures planned) had failed columns

struct ChainRec {
    int k, bs, bn, end_pos;
    int bperm[MAX_IB];
    int bkind[MAX_IB];
    double bdiag[MAX_IB], boff[MAX_IB];
    double l11[MAX_IB * MAX_IB];  // strictly lower part, zeros elsewhere, column-major
};
// Every counter on a cache line of its own: the waits poll them from many workgroups at once,
// and a line shared by several counters would queue every poll and update behind the others.
// aux is a value settled before each increment of v (the first failing column for the applied
// counters): one 8-byte load returns both, and a count seen complete comes with its final aux.
struct alignas(128) ChainCounter {
    int v;
    int aux;
    int pad[30];
};
struct ChainSync {
    ChainCounter rec;                       // inner-block records published by the leader
    ChainCounter err;                       // a wait of this front ran out
    ChainCounter applied[CHAIN_MAX_IT];     // panels done with the check of block it, and the two
                                            // wavefronts of the leader that store its tile; aux:
                                            // its first failing column (INT_MAX before)
    ChainCounter updated[CHAIN_MAX_IT];     // panels done with the updates of block it
    ChainCounter early[CHAIN_MAX_IT];       // panels that own rows of the block after the next and
                                            // have updated their first columns (no column failed)
    ChainCounter swapped[CHAIN_MAX_IT];     // panels done with their share of the failed columns' swaps
    ChainRec recs[CHAIN_MAX_IT];
};

__device__ __forceinline__ void chain_reset(ChainSync &C) {
    const int i = threadIdx.x;
    if (i == 0) { C.rec.v = 0; C.err.v = 0; }
    if (i < CHAIN_MAX_IT) {
        C.applied[i].v = 0;
        C.applied[i].aux = INT_MAX;
        C.updated[i].v = 0;
        C.early[i].v = 0;
        C.swapped[i].v = 0;
    }
}

// All threads: wait until *p >= target (thread 0 spins).  False when the front's wait ran out
// (here or in another workgroup of the front); the caller then leaves the kernel.
__device__ __forceinline__ bool chain_wait(const int *p, int target, int *err) {
    __shared__ int s_ok;
    if (threadIdx.x == 0) {
        int ok = 1;
        long long it = 0;
        while (co_ldi(p) < target) {
            if ((++it & 63) == 0 && (it > CHAIN_SPIN_LIMIT || co_ldi(err))) {
                atomicOr(err, 1);
                ok = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(4);
        }
        s_ok = ok;
    }
    __syncthreads();
    const bool ok = s_ok != 0;
    __syncthreads();  // s_ok is read by all before the next wait writes it
    return ok;
}

// chain_wait on a counter with its aux word: *aux (LDS) receives the aux read in the same 8-byte
// load that saw the count reach target.  With `also`, the same loop reads a second counter (one
// buffer load issued beside each poll, so no extra round trip) and *also_ok (LDS) tells whether it
// had reached also_target: such a count is final, a lower one says nothing.
__device__ __forceinline__ bool chain_wait_aux(ChainCounter &c, int target, int *err, int *aux,
                                               const ChainCounter *also = nullptr, int also_target = 0,
                                               int *also_ok = nullptr) {
    __shared__ int s_ok;
    if (threadIdx.x == 0) {
        int ok = 1, ao = 0;
        long long it = 0;
        unsigned long long w;
        const __amdgpu_buffer_rsrc_t ra =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<ChainCounter *>(also ? also : &c), (short)0, 64, 0x00020000);
        for (;;) {
            const int a = also ? (int)__builtin_amdgcn_raw_buffer_load_b32(ra, 0, 0, 16) : 0;
            w = __hip_atomic_load((unsigned long long *)&c.v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ao = a >= also_target;
            if ((int)(unsigned)(w & 0xffffffffu) >= target) break;
            if ((++it & 63) == 0 && (it > CHAIN_SPIN_LIMIT || co_ldi(err))) {
                atomicOr(err, 1);
                ok = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(4);
            __asm__ volatile("" ::: "memory");
        }
        *aux = (int)(unsigned)(w >> 32);
        if (also_ok) *also_ok = ao;
        s_ok = ok;
    }
    __syncthreads();
    const bool ok = s_ok != 0;
    __syncthreads();  // s_ok is read by all before the next wait writes it
    return ok;
}

// One wavefront: wait until c.v >= target; *aux receives the aux read with it.  False when the
// front's wait ran out.
__device__ __forceinline__ bool wave_poll(ChainCounter &c, int target, int *err, int *aux) {
    long long it = 0;
    for (;;) {
        const unsigned long long w =
            __hip_atomic_load((unsigned long long *)&c.v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int v = __builtin_amdgcn_readfirstlane((int)(unsigned)(w & 0xffffffffu));
        *aux = __builtin_amdgcn_readfirstlane((int)(unsigned)(w >> 32));
        if (v >= target) return true;
        if ((++it & 63) == 0 && (it > CHAIN_SPIN_LIMIT || __builtin_amdgcn_readfirstlane(co_ldi(err)))) {
            if ((threadIdx.x & 63) == 0) atomicOr(err, 1);
            return false;
        }
        __builtin_amdgcn_s_sleep(4);
        __asm__ volatile("" ::: "memory");
    }
}

// Substitution with L11 and D^-1 (factor.rs:1295-1408), four lanes per panel row: lane h of a
// row's quad holds columns 4 t + h, t = 0 .. 7, so the serial chain of 496 multiply-subtract
// pairs per row runs four columns wide and a panel's 64 rows fill the workgroup's four
// wavefronts (one row per lane kept one wavefront of four busy).  Every column receives
// its terms in ascending order, as the row form.
template <int CTRL>
__device__ __forceinline__ double quad_perm(double v) { return dpp_f64<CTRL>(v); }

template <int I, bool FULL>
struct QuadStep {
    static __device__ __forceinline__ void load(double (&c)[8], const double (*blk)[MAX_IB + 1], int h) {
#pragma unroll
        for (int t = I >> 2; t < 8; ++t) c[t] = blk[4 * t + h][I];
    }
    static __device__ __forceinline__ void run(double (&y)[8], const double (*blk)[MAX_IB + 1], int h, int bn,
                                               const double (&c0)[8], const double (&c1)[8]) {
        if constexpr (I < MAX_IB - 1) {
            if (!FULL && I >= bn) return;
            double c2[8];
            if constexpr (I + 2 < MAX_IB - 1) QuadStep<I + 2, FULL>::load(c2, blk, h);
            const double yi = quad_perm<(I & 3) * 0x55>(y[I >> 2]);
            double p[8];
#pragma unroll
            for (int t = I >> 2; t < 8; ++t) p[t] = c0[t] * yi;
#pragma unroll
            for (int t = I >> 2; t < 8; ++t) {
                const double v = y[t] - p[t];
                const bool upd = (t > (I >> 2) || h > (I & 3)) && (FULL || 4 * t + h < bn);
                y[t] = upd ? v : y[t];
            }
            __builtin_amdgcn_sched_barrier(0);
            QuadStep<I + 1, FULL>::run(y, blk, h, bn, c1, c2);
        }
    }
};

// A block's pivots as the substitution takes them: y g for a 1x1; (y a - z b) g for a 2x2, z the
// row's entry of the other column; W = L D is l d, or l d + z b.
struct PivotCoef {
    double a[MAX_IB], b[MAX_IB], g[MAX_IB], d[MAX_IB];
    int kd[MAX_IB];
    int has2;
};
// (the first wavefront; bkind .. boff in LDS)
__device__ __forceinline__ void pivot_coefs(const int8_t *bkind, const double *bdiag, const double *boff, int bn,
                                            PivotCoef &P) {
    const int c = threadIdx.x & 31;
    const int kd = c < bn ? bkind[c] : 0;
    const int f = (kd == 3 && c > 0) ? c - 1 : c, s = min(f + 1, MAX_IB - 1);  // columns of a 2x2
    const double d = bdiag[c], df = bdiag[f], ds = bdiag[s], of = boff[f];
    const double den = kd == 1 ? d : df * ds - of * of;
    const double g = 1.0 / den;
    const unsigned long long two = __ballot(kd >= 2);
    if (threadIdx.x < MAX_IB) {
        P.a[c] = kd == 2 ? ds : df;
        P.b[c] = of;
        P.g[c] = g;
        P.d[c] = d;
        P.kd[c] = kd;
        if (c == 0) P.has2 = two != 0;
    }
}

// z[t]: the entry of the other column of a 2x2 pivot (kinds kd[t])
__device__ __forceinline__ void quad_partner(const double (&y)[8], const int (&kd)[8], int h, double (&z)[8]) {
    double up[8], dn[8];  // lane h's neighbours: column c + 1 and c - 1
#pragma unroll
    for (int t = 0; t < 8; ++t) { up[t] = quad_perm<0x39>(y[t]); dn[t] = quad_perm<0x93>(y[t]); }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const double u = (h == 3) ? (t < 7 ? up[t < 7 ? t + 1 : 7] : 0.0) : up[t];
        const double l = (h == 0) ? (t > 0 ? dn[t > 0 ? t - 1 : 0] : 0.0) : dn[t];
        z[t] = (kd[t] == 2) ? u : l;
    }
}

__device__ __forceinline__ void quad_substitute(double (&y)[8], const double (*blk)[MAX_IB + 1], int bn,
                                                const PivotCoef &P) {
    const int h = fresh(threadIdx.x) & 3;
    double c0[8], c1[8];
    if (bn == MAX_IB) {
        QuadStep<0, true>::load(c0, blk, h);
        QuadStep<1, true>::load(c1, blk, h);
        QuadStep<0, true>::run(y, blk, h, bn, c0, c1);
    } else {
        QuadStep<0, false>::load(c0, blk, h);
        QuadStep<1, false>::load(c1, blk, h);
        QuadStep<0, false>::run(y, blk, h, bn, c0, c1);
    }
    int kd[8];
    double g[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) { kd[t] = P.kd[4 * t + h]; g[t] = P.g[4 * t + h]; }
    if (P.has2) {
        double z[8];
        quad_partner(y, kd, h, z);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const double v = y[t] * P.a[4 * t + h] - z[t] * P.b[4 * t + h];
            y[t] = (kd[t] >= 2) ? v * g[t] : (kd[t] == 1) ? y[t] * g[t] : y[t];
        }
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) y[t] = (kd[t] == 1) ? y[t] * g[t] : y[t];
    }
}

// W = L D of the row's entries (compute_ld_into factor.rs:1536-1563)
__device__ __forceinline__ void quad_ld(const double (&y)[8], const PivotCoef &P, double (&w)[8]) {
    const int h = fresh(threadIdx.x) & 3;
    int kd[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        kd[t] = P.kd[4 * t + h];
        w[t] = (kd[t] != 0) ? y[t] * P.d[4 * t + h] : 0.0;
    }
    if (P.has2) {
        double z[8];
        quad_partner(y, kd, h, z);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const double v = w[t] + z[t] * P.b[4 * t + h];
            w[t] = (kd[t] >= 2) ? v : w[t];
        }
    }
}

struct ChainLeaderLds {
    double blk[MAX_IB][MAX_IB + 1];      // the current block, factored (L11)
    double Ct[MAX_IB][MAX_IB + 1];       // the next block's tile, factored ahead
    double Nv[MAX_IB][MAX_IB + 1];       // that tile before its factorization
    double Wr[2 * MAX_IB][MAX_IB + 1];   // next block's L rows and W, then the factor's buffers
    double Yn[MAX_IB][MAX_IB + 1];       // next block's rows in the current block's columns
    double Cn[MAX_IB][MAX_IB + 1];       // next block's tile as it stands
    int bp[MAX_IB], nbp[MAX_IB], operm[MAX_IB], noperm[MAX_IB];
    int8_t bkind[MAX_IB], nbkind[MAX_IB];
    double bdiag[MAX_IB], boff[MAX_IB], nbdiag[MAX_IB], nboff[MAX_IB];
    PivotCoef pc;
    double wbv[1];
    int wbp[1];
    int sa[MAX_IB], sb[MAX_IB];
    SwapLds sw;
    int nsw, s_end, s_fail, s_upd, s_err;
};
constexpr int CHAIN_LC_COLS = 128;  // trailing columns per round of the panel update
struct ChainPanelLds {
    double blk[MAX_IB][MAX_IB + 1];      // L11 of the current block
    double WT[2][MAX_IB][64 + 1];        // W = L D of the panel's 64-row sub-tiles, transposed
    union {                              // one at a time, in this order within a sub-tile:
        double LT[MAX_IB][64 + 1];       //   its L in the passed columns, transposed
        double Lc[MAX_IB][MAX_IB + 1];   //   L rows of the failed block rows
        double LcT[MAX_IB][CHAIN_LC_COLS + 2];  // L rows of a round's columns, transposed
        double Yb[64][MAX_IB + 1];       // (apply) rows of a sub-tile in column order
    };
    int bp[MAX_IB];
    int8_t bkind[MAX_IB];
    double bdiag[MAX_IB], boff[MAX_IB];
    PivotCoef pc;
    int rec[4];
    int s_fail;
    int sa[MAX_IB], sb[MAX_IB], nsw;     // (failed columns)
    SwapLds sw;
};
union ChainLds {
    ChainLeaderLds ld;
    ChainPanelLds pn;
};

// A block's record (all threads; complete once every thread's stores are).
__device__ __forceinline__ void write_record(ChainRec &R, int k, int bs, int bn, int end_pos, const int *bp,
                                             const int8_t *bkind, const double *bdiag, const double *boff,
                                             const double (*blk)[MAX_IB + 1]) {
    const int tid = threadIdx.x;
    const int i = tid & (MAX_IB - 1), j0 = tid / MAX_IB;
#pragma unroll
    for (int u = 0; u < MAX_IB / 8; ++u) {
        const int j = j0 + 8 * u;
        co_std(&R.l11[i + MAX_IB * j], (j < i && i < bs) ? blk[i][j] : 0.0);
    }
    if (tid < MAX_IB) {
        co_sti(&R.bperm[tid], bp[tid]);
        co_sti(&R.bkind[tid], tid < bn ? bkind[tid] : 0);
        co_std(&R.bdiag[tid], bdiag[tid]);
        co_std(&R.boff[tid], boff[tid]);
    }
    if (tid == 64) {
        co_sti(&R.k, k);
        co_sti(&R.bs, bs);
        co_sti(&R.bn, bn);
        co_sti(&R.end_pos, end_pos);
    }
}

// The operands of the block after the current one, as threads t of nt: its rows [r0, r0 + nr) in the
// current block's columns [c0, c0 + bs) and its tile, zeros beyond.
template <int NT>
__device__ __forceinline__ void load_operands(ChainLeaderLds &L, const gdouble *A, size_t lda, const gint *perm,
                                              int c0, int bs, int r0, int nr, int t) {
    constexpr int NU = (2 * MAX_IB * MAX_IB + NT - 1) / NT;
    const __amdgpu_buffer_rsrc_t ry = co_rsrc(A + r0 + (size_t)c0 * lda), rt = co_rsrc(A + r0 + (size_t)r0 * lda);
    const unsigned l8 = (unsigned)lda * 8u;
    double v[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = t + NT * u, i = e & (MAX_IB - 1), j = (e >> 5) & (MAX_IB - 1);
        const unsigned off = 8u * i + j * l8;
        const double x = co_ldo(ry, (e < 1024 && i < nr && j < bs) ? off : CO_OOB);
        const double z = co_ldo(rt, (e >= 1024 && e < 2048 && i < nr && j <= i) ? off : CO_OOB);
        v[u] = (e < 1024) ? x : z;
    }
    const int p = (t < MAX_IB && t < nr) ? perm[r0 + t] : 0;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = t + NT * u, i = e & (MAX_IB - 1), j = (e >> 5) & (MAX_IB - 1);
        if (e < 1024) L.Yn[i][j] = v[u];
        else if (e < 2048) L.Cn[i][j] = v[u];
    }
    if (t < MAX_IB) L.noperm[t] = p;
}

// The pivot chain of a front's outer block.  Per inner block, once its record is out: substitution
// of the next block's rows and its tile's update (about 2 us each), the next block's pivots on the
// first wavefront (14 to 20 us), its record; when the panels' checks of the current block are in, the next
// record's flag goes up at once and the bookkeeping of the finished block follows.  Beside the
// pivots the other wavefronts wait for the panels' updates of the current block and bring the
// operands of the block after the next into LDS, and before them two wavefronts store the current
// block's tile while the other two substitute.  The record is written before the checks are known;
// a failed column discards it and the block factored ahead.
template <int CH>
__device__ __forceinline__ void chain_leader(FrontDev &F, AptpState &S, ChainSync &C, ChainLeaderLds &L, int nit, int NP,
                             int ib, double small) {
    const int tid = threadIdx.x;
    const int ob_start = S.ob_start;
    const int m = F.m;
    const size_t lda = m;
    gdouble *A = gbl(F.F);
    gdouble *const bk = gbl(S.backup);
    gint *const perm = gbl(F.perm);
    int k = S.kpos, end_pos = S.end_pos, nib = S.nib;
    int n1 = 0, n2 = 0;
    bool have = false;  // the current block was factored ahead; its record is out
    bool upd_prev = false;  // the panels' updates of the previous block are known complete
    int bn = 0;
    if (tid == 0) L.s_err = 0;
    for (int it = 0; it < nit; ++it) {
        const int bs = min(end_pos - k, ib);
        const int be = k + bs, nbs = min(end_pos - be, ib);
        const int ii = tid & (MAX_IB - 1), jg = tid / MAX_IB;
        if (!have) {
            // a fresh block: the panels' updates of the previous block are in place
            if (it > 0 && !upd_prev && !chain_wait(&C.updated[it - 1].v, NP, &C.err.v)) return;
            upd_prev = true;
            {
                // every load issued before any is used (one round trip)
                const __amdgpu_buffer_rsrc_t rb = co_rsrc(A + k + (size_t)k * lda);
                double v[MAX_IB / 8];
#pragma unroll
                for (int u = 0; u < MAX_IB / 8; ++u) {
                    const int j = jg + 8 * u;
                    v[u] = co_ldo(rb, (ii < bs && j <= ii) ? 8u * ii + 8u * j * (unsigned)lda : CO_OOB);
                }
#pragma unroll
                for (int u = 0; u < MAX_IB / 8; ++u) {
                    const int j = jg + 8 * u;
                    if (ii < bs && j <= ii) {
                        L.blk[ii][j] = v[u];
                        co_st(bk + ii + (size_t)j * lda, v[u]);
                    }
                }
            }
            if (tid < MAX_IB) L.operm[tid] = (tid < bs) ? perm[k + tid] : 0;
            lds_barrier();
            double bml;
            bn = block_factor_wg(L.blk, L.Wr, L.bp, L.bkind, L.bdiag, L.boff, bs, small, &bml, L.wbv, L.wbp,
                                 L.Wr + MAX_IB, [] {});
            if (tid < bn && L.bkind[tid] == 2) L.blk[tid + 1][tid] = 0.0;
            if (tid < 64) pivot_coefs(L.bkind, L.bdiag, L.boff, bn, L.pc);
            lds_barrier();
            if (bn > 0) {
                for (int j = jg; j < bs; j += 8)
                    if (ii < bs && j <= ii) co_st(A + (k + ii) + (size_t)(k + j) * lda, L.blk[ii][j]);
                if (tid < bs) perm[k + tid] = L.operm[L.bp[tid]];
            }
            if (tid == 0) atomic_max_nonneg(&F.max_l_bits, bml);
            write_record(C.recs[it], k, bs, bn, end_pos, L.bp, L.bkind, L.bdiag, L.boff, L.blk);
        }
        // the next block ahead (its operands are loaded before the record goes out: the panels
        // overwrite those rows' block entries once they have it).  A block factored ahead finds them
        // in LDS: they were left out beside its pivots only where there is no block after it
        // (nbs2 <= 0 or it + 2 >= nit there, so not `ahead` here) or where a column of the
        // block before had failed, and then it was discarded.
        const bool ahead = bs > 0 && bn == bs && nbs > 0 && it + 1 < nit;
        if (!have) {
            if (ahead) load_operands<256>(L, A, lda, perm, k, bs, be, nbs, tid);
            stores_done_barrier();
            if (tid == 0) {
                co_sti(&C.rec.v, it + 1);
                __hip_atomic_fetch_add(&C.applied[it].v, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else if (tid >= 128) {
            // the current block's tile, its backup and its rows' order: two wavefronts
            const int t = tid - 128, j0 = t / MAX_IB;
#pragma unroll
            for (int u = 0; u < MAX_IB / 4; ++u) {
                const int j = j0 + 4 * u;
                if (ii < bs && j <= ii) {
                    co_st(A + (k + ii) + (size_t)(k + j) * lda, L.blk[ii][j]);
                    co_st(bk + ii + (size_t)j * lda, L.Nv[ii][j]);
                }
            }
            if (bn > 0 && t < bs) perm[k + t] = L.operm[L.bp[t]];
            __builtin_amdgcn_s_waitcnt(0);
            if ((tid & 63) == 0) __hip_atomic_fetch_add(&C.applied[it].v, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        int bn2 = 0;
        double bml2 = 0.0, nv[MAX_IB / 8];
        if (ahead) {
            double (*Lr)[MAX_IB + 1] = L.Wr;
            double (*Wt)[MAX_IB + 1] = L.Wr + MAX_IB;
            if (tid < 128) {
                const int row = tid >> 2, h = tid & 3;
                double y[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) y[t] = L.Yn[row][L.bp[4 * t + h]];
                quad_substitute(y, L.blk, bn, L.pc);
#pragma unroll
                for (int t = 0; t < 8; ++t) Lr[row][4 * t + h] = y[t];
            }
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) L.Ct[ii][jg + 8 * u] = L.Cn[ii][jg + 8 * u];
            lds_barrier();
            if (tid < MAX_IB) L.operm[tid] = L.noperm[tid];
            next_tile_update(Lr, Wt, L.Ct, L.bkind, L.bdiag, L.boff, nbs, bs, nv);
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) L.Nv[ii][jg + 8 * u] = nv[u];
            const int be2 = be + nbs, nbs2 = min(end_pos - be2, ib);
            bn2 = block_factor_wg(L.Ct, L.Wr, L.nbp, L.nbkind, L.nbdiag, L.nboff, nbs, small, &bml2, L.wbv,
                                  L.wbp, L.Wr + MAX_IB, [&] {
                // with a failed column in the current block this block is discarded (and the panels
                // have more to do): nothing to bring
                if (nbs2 <= 0 || it + 2 >= nit) return;
                int aux;
                if (!wave_poll(C.applied[it], NP + 2, &C.err.v, &aux)) { L.s_err = 1; return; }
                if (aux < bs) return;
                // the panels that own the rows report their first columns early; with several chunks
                // per panel the whole update is awaited
                const bool single = (m - ob_start + CH - 1) / CH <= NP;
                const int own = (be2 + nbs2 - 1 - ob_start) / CH == (be2 - ob_start) / CH ? 1 : 2;
                if (!wave_poll(single ? C.early[it] : C.updated[it], single ? own : NP, &C.err.v, &aux)) {
                    L.s_err = 1;
                    return;
                }
                load_operands<192>(L, A, lda, perm, be, nbs, be2, nbs2, tid - 64);
            });
            if (tid < bn2 && L.nbkind[tid] == 2) L.Ct[tid + 1][tid] = 0.0;
            if (tid < 64) pivot_coefs(L.nbkind, L.nbdiag, L.nboff, bn2, L.pc);
            lds_barrier();
            if (L.s_err) return;
            write_record(C.recs[it + 1], be, nbs, bn2, end_pos, L.nbp, L.nbkind, L.nbdiag, L.nboff, L.Ct);
            __builtin_amdgcn_s_waitcnt(0);
        }
        // the check of block it; the panels' update count of the block comes along (complete, it
        // saves a wait).  The barriers inside complete the next record's stores.
        if (!chain_wait_aux(C.applied[it], NP + 2, &C.err.v, &L.s_fail, &C.updated[it], NP, &L.s_upd)) return;
        upd_prev = L.s_upd != 0;
        int nelim = 0;
        if (bn > 0) {
            nelim = min(L.s_fail, bn);
            if (nelim > 0 && L.bkind[nelim - 1] == 2) nelim -= 1;
        }
        const bool commit = ahead && nelim == bs;
        if (commit && tid == 0) co_sti(&C.rec.v, it + 2);
        // D and the pivot counts of the accepted columns (k_block_finish)
        if (tid < 64) {
            int is1 = 0, is2 = 0;
            if (tid < nelim) {
                const int kd = L.bkind[tid];
                const int c = k + tid;
                if (kd == 1) {
                    gbl(F.dkind)[c] = 1; gbl(F.ddiag)[c] = L.bdiag[tid]; gbl(F.doff)[c] = 0.0;
                    is1 = 1;
                } else if (kd == 2 && tid + 1 < nelim) {
                    gbl(F.dkind)[c] = 2; gbl(F.dkind)[c + 1] = 3;
                    gbl(F.ddiag)[c] = L.bdiag[tid]; gbl(F.ddiag)[c + 1] = L.bdiag[tid + 1];
                    gbl(F.doff)[c] = L.boff[tid]; gbl(F.doff)[c + 1] = 0.0;
                    is2 = 1;
                }
            }
            n1 += __popcll(__ballot(is1));
            n2 += __popcll(__ballot(is2));
        }
        if (nib < MAX_OB_IB && tid == 0) S.ib_ne[nib] = (int8_t)nelim;
        ++nib;
        if (commit) {
            if (tid == 0) atomic_max_nonneg(&F.max_l_bits, bml2);
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) L.blk[ii][jg + 8 * u] = L.Ct[ii][jg + 8 * u];
            if (tid < MAX_IB) {
                L.bp[tid] = L.nbp[tid];
                L.bkind[tid] = (tid < bn2) ? L.nbkind[tid] : 0;
                L.bdiag[tid] = L.nbdiag[tid];
                L.boff[tid] = L.nboff[tid];
            }
            lds_barrier();
            bn = bn2;
            k = be;
            have = true;
        } else {
            have = false;
            if (bn == 0 || nelim < bs) {
                // failed columns (the whole block when nothing was eliminated) move to the end of
                // the outer block, after every panel's restore and cross terms
                if (!upd_prev && !chain_wait(&C.updated[it].v, NP, &C.err.v)) return;
                upd_prev = true;
                if (tid == 0) {
                    L.nsw = failed_swaps(k, bs, bn, nelim, end_pos, L.sa, L.sb);
                    L.s_end = end_pos;
                }
                __syncthreads();
                end_pos = L.s_end;
                if (L.nsw > 0) {
                    apply_swaps_shared(F, S, L.sa, L.sb, L.nsw, L.sw, -1, NP);
                    if (!chain_wait(&C.swapped[it].v, NP, &C.err.v)) return;
                }
            }
            k += nelim;
        }
    }
    if (tid == 0) {
        S.kpos = k;
        S.end_pos = end_pos;
        S.nib = nib;
        S.fail_min = INT_MAX;
        S.pref = 0;
        S.nx_valid = 0;
        F.n1 += n1;
        F.n2 += n2;
    }
}

// Columns [c0, c0 + ncol) of the L rows of an update round, transposed into LDS: the loads (cl_load,
// in flight as long as the caller likes) and the LDS stores.
constexpr int CHAIN_NL = CHAIN_LC_COLS * MAX_IB / 256;
__device__ __forceinline__ void cl_load(double (&v)[CHAIN_NL], const gdouble *A, size_t lda, int c0, int ncol, int k,
                                        int nelim) {
    // thread: column tid % 128, elimination steps j = tid / 128 + 2 u; outside: past the range, zero
    static_assert(CHAIN_LC_COLS == 128, "thread layout of a round's L rows");
    const __amdgpu_buffer_rsrc_t rb = co_rsrc(A + c0 + (size_t)k * lda);
    const int tid = fresh(threadIdx.x), l8 = fresh_uniform((int)lda * 8);
    const int cc = tid & 127, jh = tid >> 7;
    const unsigned off = cc * 8 + jh * l8;
#pragma unroll
    for (int u = 0; u < CHAIN_NL; ++u) {
        const unsigned o = off + 2 * u * l8;
        v[u] = co_ldo(rb, (cc < ncol && 2 * u + jh < nelim) ? o : CO_OOB);
    }
}
__device__ __forceinline__ void cl_store(const double (&v)[CHAIN_NL], double (*LcT)[CHAIN_LC_COLS + 2]) {
    const int tid = fresh(threadIdx.x), cc = tid & 127, jh = tid >> 7;
#pragma unroll
    for (int u = 0; u < CHAIN_NL; ++u) LcT[2 * u + jh][cc] = v[u];
}

// Update round: thread (tx, ty) holds rows R0 + tx + 16 i (i < 4) x columns c0 + 4 ty + q + 64 p
// (q < 4, p < 2) of the front in cv; each sum runs over j ascending from zero.
__device__ __forceinline__ void cu_load(double (&cv)[4][8], __amdgpu_buffer_rsrc_t rc, size_t lda, bool on = true) {
    const int tid = fresh(threadIdx.x), l8 = fresh_uniform((int)lda * 8);
    const int tx = tid & 15, ty = tid >> 4;
    const unsigned vo = on ? (unsigned)(tx * 8 + 4 * ty * l8) : CO_OOB;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const unsigned o = vo + ((q & 3) + 64 * (q >> 2)) * l8;
#pragma unroll
        for (int i = 0; i < 4; ++i) cv[i][q] = co_ldo(rc, o + 128 * i);
    }
}
__device__ __forceinline__ void cu_sums(double (&acc)[4][8], const double (*WT)[64 + 1],
                                        const double (*LcT)[CHAIN_LC_COLS + 2], int nelim) {
    const int tid = fresh(threadIdx.x), tx = tid & 15, ty = tid >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[i][q] = 0.0;
    auto step = [&](int j) {
        double wv[4], lc[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) wv[i] = WT[j][tx + 16 * i];
#pragma unroll
        for (int q = 0; q < 8; ++q) lc[q] = LcT[j][4 * ty + (q & 3) + 64 * (q >> 2)];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[i][q] += wv[i] * lc[q];
    };
    if (nelim == MAX_IB) {
#pragma unroll 4
        for (int j = 0; j < MAX_IB; ++j) step(j);
    } else {
        for (int j = 0; j < nelim; ++j) step(j);
    }
}
// rows >= be below r1, lower triangle; the leader's tile (rows and columns below lead) left out
__device__ __forceinline__ void cu_store(const double (&cv)[4][8], const double (&acc)[4][8],
                                         __amdgpu_buffer_rsrc_t rc, size_t lda, int R0, int r1, int c0, int ncol,
                                         int be, int lead) {
    const int tid = fresh(threadIdx.x), l8 = fresh_uniform((int)lda * 8);
    const int tx = tid & 15, ty = tid >> 4;
    const int vo = tx * 8 + 4 * ty * l8;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int cc = 4 * ty + (q & 3) + 64 * (q >> 2), col = c0 + cc;
        const int o = vo + ((q & 3) + 64 * (q >> 2)) * l8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = R0 + tx + 16 * i;
            const bool ok = r >= be && r < r1 && cc < ncol && r >= col && !(r < lead && col < lead);
            co_stb(rc, ok ? (unsigned)(o + 128 * i) : CO_OOB, cv[i][q] - acc[i][q]);
        }
    }
}

// A block's failed columns move to the end of the outer block: the panel's share of the lines, after
// every panel's restore and cross terms.  False when a wait ran out.
__device__ __attribute__((noinline)) bool chain_panel_failed(FrontDev &F, AptpState &S, ChainSync &C, ChainPanelLds &L,
                                                             int it, int k, int bs, int bn, int nelim, int end_pos,
                                                             int pidx, int NP) {
    if (threadIdx.x == 0) L.nsw = failed_swaps(k, bs, bn, nelim, end_pos, L.sa, L.sb);
    __syncthreads();
    if (L.nsw == 0) return true;
    if (!chain_wait(&C.updated[it].v, NP, &C.err.v)) return false;
    apply_swaps_shared(F, S, L.sa, L.sb, L.nsw, L.sw, pidx, NP);
    if (threadIdx.x == 0) __hip_atomic_fetch_add(&C.swapped[it].v, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Panel rows of chunk c: [ob_start + c * CH, min(ob_start + (c + 1) * CH, m)).
//
// The chain of one inner block through a panel is latency: device-scope loads of 1-3 us each and
// the signals between workgroups.  With one chunk per panel (every level without delays) and no
// failed column, W = L D goes from the substitution's registers straight to LDS, the columns to
// update are loaded before the wait for the other panels' checks, the L rows of the second round
// of columns during the first round's products, and the row permutation of earlier columns runs
// after the panel has reported: a block's update takes 16.4 us from 28.4 (64^3 Helmholtz), 10.8
// from 21.8 (40^3).
template <int CH>
__device__ __forceinline__ void chain_panel(FrontDev &F, AptpState &S, ChainSync &C, ChainPanelLds &L, int pidx, int NP, int nit,
                            int ib, double threshold) {
    static_assert(CH == 64 || CH == 128, "panel rows per workgroup: 64 or 128 (the apply's LDS rows)");

    const int m = F.m;
    gdouble *A = gbl(F.F);
    gdouble *const bk = gbl(S.backup);
    const int ob_start = S.ob_start, obe = S.ob_start + S.ob_cols;
    const int nchunk = (m - ob_start + CH - 1) / CH;
    const bool single = nchunk <= NP;  // at most one chunk per panel
    const double bound = 1.0 / threshold;
    constexpr int NS = CH / 64;  // sub-tiles of a chunk; thread (row = tid / 4, h = tid % 4) of each
    double y[NS][8];             // columns 4 t + h of the row's block entries
    int pre_k = -1, pre_bs = 0;  // block whose rows are in y already
    // a chunk's block entries in column order (zeros outside the front's live rows and beyond the
    // block, by the resource's range)
    auto load_rows = [&](int c, int k, int bs) {
        const int t4 = fresh(threadIdx.x), row = t4 >> 2, h = t4 & 3;
        const unsigned l8 = (unsigned)fresh_uniform(m * 8);
        const __amdgpu_buffer_rsrc_t rb = co_rsrc(A + (size_t)k * m);
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            const int r = ob_start + c * CH + 64 * u + row;
            const unsigned off = (r >= k + bs && r < m) ? 8u * r + h * l8 : CO_OOB;
#pragma unroll
            for (int t = 0; t < 8; ++t) y[u][t] = co_ldo(rb, 4 * t + h < bs ? off + 4 * t * l8 : CO_OOB);
        }
    };
    for (int it = 0; it < nit; ++it) {
        if (!chain_wait(&C.rec.v, it + 1, &C.err.v)) return;
        const int tid = fresh(threadIdx.x);
        const size_t lda = (size_t)(unsigned)fresh_uniform(m);
        const ChainRec &R = C.recs[it];
        {
            double v[MAX_IB / 8];
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) v[u] = co_ldo(co_rsrc(gbl(R.l11)), 8u * (tid + 256 * u));
            if (tid < 64) {
                const __amdgpu_buffer_rsrc_t ri = co_rsrc((const gdouble *)gbl(&R.k));
                const int c = tid & 31;
                const int p = __builtin_amdgcn_raw_buffer_load_b32(ri, 16 + 4 * c, 0, 16);
                const int kd = __builtin_amdgcn_raw_buffer_load_b32(ri, 16 + 4 * MAX_IB + 4 * c, 0, 16);
                const double dg = co_ldo(ri, 16 + 8 * MAX_IB + 8 * c);
                const double of = co_ldo(ri, 16 + 16 * MAX_IB + 8 * c);
                const int hd = __builtin_amdgcn_raw_buffer_load_b32(ri, 4 * (c & 3), 0, 16);
                L.bp[c] = p;
                L.bkind[c] = (int8_t)kd;
                L.bdiag[c] = dg;
                L.boff[c] = of;
                L.rec[c & 3] = hd;
                wave_sync();
                pivot_coefs(L.bkind, L.bdiag, L.boff, MAX_IB, L.pc);  // (kind 0 beyond the eliminated columns)
            }
            const int i = tid & (MAX_IB - 1), j0 = tid / MAX_IB;
#pragma unroll
            for (int u = 0; u < MAX_IB / 8; ++u) L.blk[i][j0 + 8 * u] = v[u];
        }
        lds_barrier();
        const int k = __builtin_amdgcn_readfirstlane(L.rec[0]), bs = __builtin_amdgcn_readfirstlane(L.rec[1]);
        const int bn = __builtin_amdgcn_readfirstlane(L.rec[2]), end_pos = __builtin_amdgcn_readfirstlane(L.rec[3]);
        const int be = k + bs;
        // the panel's one chunk has rows below the block: its update takes the short path when
        // the block has no failed column
        const int r0p = ob_start + pidx * CH, r1p = min(r0p + CH, m);
        const bool fast = single && pidx < nchunk && r1p > be && bn == bs;
        if (bn > 0) {
            if (pre_k != k || pre_bs != bs) load_rows(pidx, k, bs);
            for (int c = pidx; c < nchunk; c += NP) {
                if (c != pidx) load_rows(c, k, bs);
                const int row = tid >> 2, h = tid & 3;
                const unsigned l8 = (unsigned)fresh_uniform((int)lda * 8);
                int first = INT_MAX;
#pragma unroll
                for (int u = 0; u < NS; ++u) {
                    const int rb0 = ob_start + c * CH + 64 * u, r = rb0 + row;
                    if (rb0 + 63 < be || rb0 >= m) continue;  // (uniform)
                    const bool live = r >= be && r < m;
                    // backed up as they are (restore_diagonal_with_perm reads the backup in
                    // column order), then gathered into pivot order through LDS rows of the
                    // wavefront's own (its LDS operations are performed in order)
                    const __amdgpu_buffer_rsrc_t rk = co_rsrc(bk), ra = co_rsrc(A + (size_t)k * lda);
                    const unsigned ok = live ? 8u * (r - k) + h * l8 : CO_OOB, oa = live ? 8u * r + h * l8 : CO_OOB;
                    double *yb = L.Yb[row];
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        co_stb(rk, 4 * t + h < bs ? ok + 4 * t * l8 : CO_OOB, y[u][t]);
                        yb[4 * t + h] = y[u][t];
                    }
                    wave_sync();
#pragma unroll
                    for (int t = 0; t < 8; ++t) y[u][t] = yb[L.bp[4 * t + h]];
                    wave_sync();
                    quad_substitute(y[u], L.blk, bn, L.pc);
#pragma unroll
                    for (int t = 7; t >= 0; --t) {
                        const int q = 4 * t + h;
                        co_stb(ra, q < bs ? oa + 4 * t * l8 : CO_OOB, y[u][t]);
                        if (live && q < bn && fabs(y[u][t]) >= bound) first = min(first, L.pc.kd[q] == 3 ? q - 1 : q);
                    }
                }
                first = wave_min_int(first);
                if ((tid & 63) == 0 && first != INT_MAX) atomicMin(&C.applied[it].aux, first);
            }
        }
        stores_done_barrier();
        if (tid == 0) __hip_atomic_fetch_add(&C.applied[it].v, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        double pml = 0.0;  // (fast) the thread's largest |l|
        if (fast) {
            // W = L D, used if no column fails
#pragma unroll
            for (int u = 0; u < NS; ++u) {
                double w[8];
                quad_ld(y[u], L.pc, w);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    L.WT[u][4 * t + (tid & 3)][tid >> 2] = w[t];
                    pml = max_abs(pml, y[u][t]);
                }
            }
        }
        // (fast) the first round's columns of the first sub-tile: this panel's own rows
        double cv[4][8];
        const int R0f = (r0p + 63 < be) ? r0p + 64 : r0p;  // first sub-tile with rows below the block
        __amdgpu_buffer_rsrc_t rc = co_rsrc_front(A, lda, (size_t)min(R0f, m - 1) + (size_t)min(be, m - 1) * lda);
        cu_load(cv, rc, lda, fast && be < obe);
        if (!chain_wait_aux(C.applied[it], NP + 2, &C.err.v, &L.s_fail)) return;
        int permute_from = -1, nel = 0;
        if (bn > 0) {
            int nelim = min(L.s_fail, bn);
            if (nelim > 0 && L.bkind[nelim - 1] == 2) nelim -= 1;
            nelim = __builtin_amdgcn_readfirstlane(nelim);
            nel = nelim;
            const int nbs = min(end_pos - be, ib);
            const bool ahead = nelim == bs && nbs > 0 && it + 1 < nit;
            const int lead = ahead ? be + nbs : be;
            const int be2 = be + nbs, nbs2 = min(end_pos - be2, ib);
            const int nf = bs - nelim;
            double ml = 0.0;
            // a panel without rows below the block has nothing to do when no column failed
            const bool idle = single && nf == 0 && (pidx >= nchunk || r1p <= be);
            if (fast && nf == 0) {
                ml = pml;
                // rounds (sub-tile, 128 columns); a round's columns are loaded at the end of the one
                // before it
                int R0 = R0f, c0 = be;
                double lv[CHAIN_NL];
                cl_load(lv, A, lda, be, min(CHAIN_LC_COLS, obe - be), k, nelim);
                while (R0 < r1p && c0 < obe) {
                    const int ncol = min(CHAIN_LC_COLS, obe - c0);
                    int R1 = R0, c1 = c0 + CHAIN_LC_COLS;
                    if (c1 >= obe || R0 + 63 < c1) { R1 = R0 + 64; c1 = be; }  // no row reaches the columns from c1
                    const bool more = R1 < r1p;
                    __syncthreads();  // the previous round's LDS reads are done
                    cl_store(lv, L.LcT);
                    cl_load(lv, A, lda, more ? c1 : be, more ? min(CHAIN_LC_COLS, obe - c1) : 0, k, nelim);
                    __syncthreads();
                    double acc[4][8];
                    cu_sums(acc, L.WT[(R0 - r0p) >> 6], L.LcT, nelim);
                    cu_store(cv, acc, rc, lda, R0, r1p, c0, ncol, be, lead);
                    if (ahead && c0 == be && R0 < be2 + nbs2 && min(R0 + 64, r1p) > be2 && (R0 + 64 >= be2 + nbs2 || R0 + 64 >= r1p)) {
                        // (uniform) the leader's operands: rows of the block after the next, the last
                        // of this panel's sub-tiles that hold some
                        stores_done_barrier();
                        if (tid == 0)
                            __hip_atomic_fetch_add(&C.early[it].v, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    R0 = R1;
                    c0 = c1;
                    if (!more) break;
                    rc = co_rsrc_front(A, lda, (size_t)R0 + (size_t)c0 * lda);
                    cu_load(cv, rc, lda);
                }
            }
            // 64-row sub-tiles of the panel's rows at or below the block
            for (int c = (fast && nf == 0) || idle ? nchunk : pidx; c < nchunk; c += NP) {
                const int r0c = ob_start + c * CH, r1 = min(r0c + CH, m);
                for (int R0 = r0c; R0 < r1; R0 += 64) {
                    if (R0 + 64 <= k) continue;  // (uniform)
                    __syncthreads();             // the previous sub-tile's LDS reads are done
                    // L rows of the sub-tile in the passed columns -> LT[j][row]; W = L D
                    // (ld_entry, compute_ld_into factor.rs:1536-1563) -> WT[j][row]
                    double (*WT)[64 + 1] = L.WT[0];
                    {
                        const int rr = tid & 63, jg = tid >> 6, r = R0 + rr;
                        const bool valid = r >= k && r < r1;
                        double lv[MAX_IB / 4];
                        const __amdgpu_buffer_rsrc_t rb = co_rsrc(A + (size_t)k * lda);
                        const size_t ro = (size_t)min(r, m - 1);
#pragma unroll
                        for (int u = 0; u < MAX_IB / 4; ++u) {
                            const int j = jg + 4 * u;
                            const double v = co_ldb(rb, ro + (size_t)(j < nelim ? j : 0) * lda);
                            lv[u] = (valid && j < nelim) ? v : 0.0;
                        }
#pragma unroll
                        for (int u = 0; u < MAX_IB / 4; ++u) {
                            L.LT[jg + 4 * u][rr] = lv[u];
                            // max |L| over the passed columns of the rows below the block
                            if (valid && r >= be && fabs(lv[u]) > ml) ml = fabs(lv[u]);
                        }
                    }
                    __syncthreads();
                    {
                        const int rr = tid & 63, jg = tid >> 6;
#pragma unroll
                        for (int u = 0; u < MAX_IB / 4; ++u) {
                            const int j = jg + 4 * u;
                            // the three forms side by side, one selected
                            const int kd = L.bkind[j];
                            const double dj = L.bdiag[j];
                            const double lj = L.LT[j][rr];
                            const double v1 = lj * dj;
                            const double v2 = lj * dj + L.LT[j + 1 < MAX_IB ? j + 1 : j][rr] * L.boff[j];
                            const double v3 = L.LT[j > 0 ? j - 1 : 0][rr] * L.boff[j > 0 ? j - 1 : 0] + lj * dj;
                            const double v = (kd == 1) ? v1 : (kd == 2) ? v2 : (kd == 3) ? v3 : 0.0;
                            WT[j][rr] = (j < nelim) ? v : 0.0;
                        }
                    }
                    __syncthreads();
                    // partial restore and cross terms of the failed columns (factor.rs:1962-2008)
                    if (nf > 0) {
                        {
                            const int jf = tid & 31, c0 = tid >> 5;
                            double v[MAX_IB / 8];
#pragma unroll
                            for (int u = 0; u < MAX_IB / 8; ++u) {
                                const int cc = c0 + 8 * u;
                                v[u] = (jf < nf && cc < nelim) ? co_ld(A + (k + nelim + jf) + (size_t)(k + cc) * lda) : 0.0;
                            }
#pragma unroll
                            for (int u = 0; u < MAX_IB / 8; ++u) L.Lc[jf][c0 + 8 * u] = v[u];
                        }
                        __syncthreads();
                        const int rr = tid & 63, g = tid >> 6, r = R0 + rr;
                        if (r >= k && r < r1) {
                            gdouble *row = A + r;
                            for (int j = nelim + g; j < bs; j += 4) {
                                const size_t cj = (size_t)(k + j) * lda;
                                double v = 0.0;
                                bool have_v = false;
                                if (nelim < bn) {
                                    if (r < be) {
                                        const int i = r - k;
                                        if (i >= j) {
                                            const int br = L.bp[i], bc = L.bp[j];
                                            v = (br >= bc) ? co_ld(bk + br + (size_t)bc * lda) : co_ld(bk + bc + (size_t)br * lda);
                                            have_v = true;
                                        }
                                    } else {
                                        v = co_ld(bk + (r - k) + (size_t)L.bp[j] * lda);
                                        have_v = true;
                                    }
                                }
                                if (nelim > 0) {
                                    const int jf = j - nelim;
                                    if (r >= be || r - k - nelim >= jf) {
                                        double sx = 0.0;
                                        for (int c2 = 0; c2 < nelim; ++c2) sx += WT[c2][rr] * L.Lc[jf][c2];
                                        if (!have_v) v = co_ld(row + cj);
                                        v = v - sx;
                                        have_v = true;
                                    }
                                }
                                if (have_v) co_st(row + cj, v);
                            }
                        }
                    }
                    // trailing columns of the outer block, CHAIN_LC_COLS per round, the round's L
                    // rows staged transposed in LDS
                    if (nelim == 0 || R0 + 63 < be) continue;  // (uniform)
                    for (int c0 = be; c0 < obe; c0 += CHAIN_LC_COLS) {
                        const int ncol = min(CHAIN_LC_COLS, obe - c0);
                        if (R0 + 63 < c0) break;  // (uniform) no row of the sub-tile reaches them
                        __syncthreads();
                        rc = co_rsrc_front(A, lda, (size_t)R0 + (size_t)c0 * lda);
                        {
                            double lv[CHAIN_NL];
                            cl_load(lv, A, lda, c0, ncol, k, nelim);
                            cl_store(lv, L.LcT);
                        }
                        __syncthreads();
                        double cs[4][8], acc[4][8];
                        cu_load(cs, rc, lda);
                        cu_sums(acc, WT, L.LcT, nelim);
                        cu_store(cs, acc, rc, lda, R0, r1, c0, ncol, be, lead);
                    }
                }
            }
            ml = wave_fmax(ml);
            if ((tid & 63) == 0) atomic_max_nonneg(&F.max_l_bits, ml);
            permute_from = nf;
        }
        // block rows permuted in the columns factored before this block, this panel's share: with
        // failed columns before the panel reports (the leader then moves some of these rows), else
        // after (the rows are final)
        auto permute_rows = [&]() -> bool {
            if (k == 0 || bs <= 0) return true;
            // a panel may still read these rows for its update by the block before
            if (it > 0 && !chain_wait(&C.updated[it - 1].v, NP, &C.err.v)) return false;
            const int per = (k + NP - 1) / NP;
            const int cb = pidx * per, ce = min(k, cb + per);
            const int i = tid & 31, half = (tid >> 5) & 1, wv = tid >> 6;
            if (i < bs) {
                const int sr = L.bp[i];
                // 128 columns per step, all loads issued before the stores
                for (int cs = cb; cs < ce; cs += 128) {
                    const __amdgpu_buffer_rsrc_t rb = co_rsrc(A + k + (size_t)cs * lda);
                    double v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int cc = 2 * wv + half + 8 * u;  // column cs + cc
                        const double x = co_ldb(rb, (size_t)sr + (size_t)(cs + cc < ce ? cc : 0) * lda);
                        v[u] = x;
                    }
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int c = cs + 2 * wv + half + 8 * u;
                        if (c < ce) co_st(A + (k + i) + (size_t)c * lda, v[u]);
                    }
                }
            }
            return true;
        };
        if (permute_from > 0 && !permute_rows()) return;
        stores_done_barrier();
        if (tid == 0) __hip_atomic_fetch_add(&C.updated[it].v, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // without failed columns nothing moves: the next block starts at be, its rows can come now
        pre_k = -1;
        if (nel < bs) {
            if (!chain_panel_failed(F, S, C, L, it, k, bs, bn, nel, end_pos, pidx, NP)) return;
            continue;
        }
        if (permute_from == 0 && single && pidx < nchunk && it + 1 < nit && end_pos > be) {
            pre_k = be;
            pre_bs = min(end_pos - be, ib);
            load_rows(pidx, pre_k, pre_bs);
        }
        if (permute_from == 0 && !permute_rows()) return;
    }
}

// One outer block of every listed front: item (APTP slot, role, front, NP); role 0 = leader,
// role 1 + p = panel p of NP.
template <int CH>
__global__ __launch_bounds__(256, 2) void k_aptp_outer(FrontDev *__restrict__ fr, AptpState *__restrict__ st,
                                                    ChainSync *__restrict__ cs, const int4 *__restrict__ items,
                                                    int nb, int ib, double small, double threshold) {
    __shared__ ChainLds lds;
    const int4 itm = items[blockIdx.x];
    FrontDev &F = fr[itm.z];
    AptpState &S = st[itm.x];
    ChainSync &C = cs[itm.x];
    const int nit = (S.ob_cols + ib - 1) / ib;
    if (itm.y == 0) {
        chain_leader<CH>(F, S, C, lds.ld, nit, itm.w, ib, small);
        if (threadIdx.x == 0 && co_ldi(&C.err.v)) atomicOr(&F.flags, FRONT_CHAIN_ERR);
    } else {
        chain_panel<CH>(F, S, C, lds.pn, itm.y - 1, itm.w, nit, ib, threshold);
    }
}

// Start of an outer block (two_level_factor, factor.rs:2126-2131); ob == 0 also initialises.
__device__ void outer_begin(FrontDev &F, AptpState &S, int ob, int nb, int ib) {
    const int p = F.k;
    const bool two = p > nb;
    const int nouter = two ? (p + nb - 1) / nb : 1;
    if (ob >= nouter) return;
    if (threadIdx.x == 0) {
        if (ob == 0) { S.gne = 0; S.remaining = p; }
        S.ob_start = S.gne;
        S.ob_cols = two ? min(S.remaining, nb) : p;
        S.kpos = S.ob_start;
        S.end_pos = S.ob_start + S.ob_cols;
        S.nib = 0;
        S.pref = 0;
        S.nx_valid = 0;
    }
    __syncthreads();
    copy_next_block(F, S, ib);
}

// End of an outer block: failed columns move to the end of the remaining fully-summed
// region (factor.rs:2195-2206), counters advance; the last block records ne.  Returns false
// when the front has no outer block ob or only one outer block (then it has no block ob + 1
// either); the return is the same for every thread of the workgroup.  A front that ends with columns
// left over joins the list `left` (its length, then the fronts) that k_tpp_left works through.
__device__ bool outer_end(FrontDev *__restrict__ fr, int front, AptpState &S, int ob, int nb, int la,
                          int *__restrict__ left) {
    FrontDev &F = fr[front];
    auto last = [&](int ne) {
        F.ne = ne;
        if (ne < F.k) left[1 + atomicAdd(left, 1)] = front;
    };
    const bool deferred = !(F.flags & FRONT_ALLFS);
    const int p = F.k;
    const bool two = p > nb;
    const int nouter = two ? (p + nb - 1) / nb : 1;
    if (ob >= nouter) return false;
    __shared__ int sa[MAX_IB], sb[MAX_IB];
    __shared__ SwapLds sw;
    __shared__ int nsw;
    const int tid = threadIdx.x;
    if (!two) {
        if (tid == 0) last(S.kpos);
        return false;
    }
    const int obne = S.kpos - S.ob_start;
    const int nfail = S.ob_cols - obne;
    if (nfail > 0 && tid == 0) {
        F.obfail |= 1ull << min(ob, 63);
        // the trailing update of this block was planned to run beside the next block, which
        // is only correct without the delay swaps below: the factorization is repeated
        if (la) atomicOr(&F.flags, FRONT_LA_ERR);
    }
    if (deferred && tid == 0) {
        // algorithmic flops of this block's outer update (k_schur mode 1): 2 obne per entry of
        // the lower trapezoid rows [r0, m) x columns [r0, p)
        const double r0 = S.ob_start + S.ob_cols, nr = F.m - r0, nc = p - r0;
        if (obne > 0 && nc > 0) F.uflops += 2.0 * obne * (nc * (nc + 1.0) / 2.0 + (nr - nc) * nc);
    }
    // process the swap sequence in pieces of at most MAX_IB swaps (<= 2*MAX_IB lines)
    int done = 0;
    while (done < nfail) {
        const int cnt_sw = min(MAX_IB, nfail - done);
        if (tid == 0) {
            int n = 0;
            for (int i = done; i < done + cnt_sw; ++i) {
                const int fp = S.ob_start + obne + i;
                const int end = S.ob_start + S.remaining - 1 - i;
                if (fp < end) { sa[n] = fp; sb[n] = end; ++n; }
            }
            nsw = n;
        }
        __syncthreads();
        apply_swaps(F, S, sa, sb, nsw, sw);
        done += cnt_sw;
    }
    __syncthreads();
    if (tid == 0) {
        S.gne += obne;
        S.remaining -= S.ob_cols;
        if (ob == nouter - 1) last(S.gne);
    }
    return true;
}

// The first outer block of every front of a level: the APTP state is installed from its staged
// initial value (scratch pointers, fail_min = INT_MAX, the rest zero), then outer block 0 starts.
// Clears the list of fronts with columns left over.
__global__ __launch_bounds__(256) void k_outer_first(FrontDev *__restrict__ fr,
                                                     AptpState *__restrict__ st,
                                                     const AptpState *__restrict__ init,
                                                     const int *__restrict__ flist, int nb, int ib,
                                                     ChainSync *__restrict__ cs, int *__restrict__ left) {
    if (cs) chain_reset(cs[blockIdx.x]);
    if (blockIdx.x == 0 && threadIdx.x == 0) *left = 0;
    FrontDev &F = fr[flist[blockIdx.x]];
    AptpState &S = st[blockIdx.x];
    const AptpState &I = init[blockIdx.x];
    static_assert(sizeof(AptpState) % sizeof(int) == 0, "AptpState copied as ints");
    const int *src = (const int *)&I;
    int *dst = (int *)&S;
    for (int i = threadIdx.x; i < (int)(sizeof(AptpState) / sizeof(int)); i += blockDim.x) dst[i] = src[i];
    __syncthreads();
    outer_begin(F, S, 0, nb, ib);
}

__global__ __launch_bounds__(256) void k_outer_end(FrontDev *__restrict__ fr,
                                                   AptpState *__restrict__ st,
                                                   const int *__restrict__ flist, int ob, int nb,
                                                   int *__restrict__ left) {
    outer_end(fr, flist[blockIdx.x], st[blockIdx.x], ob, nb, 0, left);
}

// The end of outer block ob and the start of ob + 1 in one launch (one workgroup per front).
// la: block ob's trailing update runs beside this launch and block ob + 1 (planned without failed
// columns in block ob).
__global__ __launch_bounds__(512) void k_outer_next(FrontDev *__restrict__ fr,
                                                    AptpState *__restrict__ st,
                                                    const int *__restrict__ flist, int ob, int nb,
                                                    int ib, ChainSync *__restrict__ cs, int la,
                                                    int *__restrict__ left) {
    if (cs) chain_reset(cs[blockIdx.x]);
    const int front = flist[blockIdx.x];
    AptpState &S = st[blockIdx.x];
    if (!outer_end(fr, front, S, ob, nb, la, left)) return;
    __syncthreads();
    outer_begin(fr[front], S, ob + 1, nb, ib);
}

// ===========================================================================
// Threshold partial pivoting (tpp_factor / tpp_factor_rect, factor.rs:2268-2947).
// Of whole fronts (k_tpp) or of the columns that APTP left over (k_tpp_left).
// ===========================================================================
// Raw buffer loads (gfx9 resource: stride 0, range-checked against num_records): an offset at or
// beyond the range loads zero without touching memory.
constexpr unsigned BUF_RANGE = 0x7FFFFFF0u;
constexpr unsigned BUF_OOB = 0x7FFFFFF8u;  // outside every resource made by buf_rsrc
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)BUF_RANGE, 0x00020000);
}
__device__ __forceinline__ float buf_load_f32(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
__device__ __forceinline__ double buf_load_f64(__amdgpu_buffer_rsrc_t r, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

// Reductions over one wavefront (every lane active), the result in all lanes.  max_abs: magnitudes,
// NaN ignored.
__device__ __forceinline__ double wave_max_abs(double v) {
    v = max_abs(v, dpp_f64<0xB1>(v));
    v = max_abs(v, dpp_f64<0x4E>(v));
    v = max_abs(v, dpp_f64<0x141>(v));
    v = max_abs(v, dpp_f64<0x140>(v));
    return max_abs(max_abs(readlane_f64(v, 0), readlane_f64(v, 16)), max_abs(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// A front from its first uneliminated column on, in local indices: m rows, n fully-summed columns,
// lower triangle, column-major.  P: LDS (a staged front) or global memory.
template <class P>
struct TppMat {
    P A;
    size_t ld;
    int m, n;
    __device__ __forceinline__ size_t at(int r, int q) const {
        return (r >= q) ? r + q * ld : q + r * ld;
    }
};

// Pivot tests by one wavefront each (threshold partial pivoting's candidates are independent until
// one is taken, so a workgroup tests as many at once as it has wavefronts).
constexpr int TPP_B = 4;  // entries per lane whose loads are issued together (a line below 256: one batch)

// max |entry| of line (row part left of it, column part below it) from index `from`, without the
// diagonal and index ex; NaN ignored, 0 when there is none.  *big: one of them is >= small.
template <class P>
__device__ __forceinline__ double tpp_line_max(const TppMat<P> &M, int line, int from, int ex, double small = 0.0,
                                               bool *big = nullptr) {
    const int lane = threadIdx.x & 63;
    double best = 0.0;
    bool b = false;
    for (int q0 = from + lane; q0 < M.m; q0 += 64 * TPP_B) {
        double v[TPP_B];
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) v[t] = M.A[M.at(line, min(q0 + 64 * t, M.m - 1))];
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) {
            const int q = q0 + 64 * t;
            const bool in = q < M.m && q != line && q != ex;
            best = in ? max_abs(best, v[t]) : best;
            b |= in && fabs(v[t]) >= small;
        }
    }
    if (big) *big = __any(b);
    return wave_max_abs(best);
}

__device__ __forceinline__ bool tpp_test_2x2(double a11, double a21, double a22, double maxt, double maxp, double u,
                                             double small) {
    const double maxpiv = fmax(fmax(fabs(a11), fabs(a21)), fabs(a22));
    if (maxpiv < small) return false;
    const double detscale = 1.0 / maxpiv;
    const double d0 = (a11 * detscale) * a22;
    const double d1 = (a21 * detscale) * a21;
    const double det = d0 - d1;
    if (fabs(det) < fmax(fmax(small, fabs(d0 / 2.0)), fabs(d1 / 2.0))) return false;
    const double i11 = (a22 * detscale) / det;
    const double i12 = (-a21 * detscale) / det;
    const double i22 = (a11 * detscale) / det;
    if (fmax(maxt, maxp) < small) return true;
    const double x1 = fabs(i11) * maxt + fabs(i12) * maxp;
    const double x2 = fabs(i12) * maxt + fabs(i22) * maxp;
    return u * fmax(x1, x2) < 1.0;
}

enum { TPP_NONE = 0, TPP_ZERO = 1, TPP_2X2 = 2, TPP_1X1 = 3 };

// Candidate p (> from) of a step at column `from`: a column without an entry of magnitude >= small,
// a 2x2 with t, the largest entry of its row among [from, p) (the first of equals), or a 1x1.
template <class P>
__device__ __forceinline__ int tpp_candidate(const TppMat<P> &M, int p, int from, double u, double small, int *tout) {
    const int lane = threadIdx.x & 63;
    // one pass over the line: per lane the row part's largest entry (first index), the largest of
    // the rest kept per entry for the exclusion of t
    double bv = -1.0, oth = 0.0;
    int bi = INT_MAX;
    bool big = false;
    for (int q0 = from + lane; q0 < M.m; q0 += 64 * TPP_B) {
        double v[TPP_B];
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) v[t] = fabs(M.A[M.at(p, min(q0 + 64 * t, M.m - 1))]);
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) {
            const int q = q0 + 64 * t;
            const bool row = q < p, up = row && v[t] > bv;
            const double lose = up ? bv : v[t];  // what is not the lane's best of the row part
            big |= q < M.m && v[t] >= small;
            oth = (q != p && q < M.m && lose > oth) ? lose : oth;
            bi = up ? q : bi;
            bv = up ? v[t] : bv;
        }
    }
    if (!__any(big)) return TPP_ZERO;
    const double bm = wave_max_abs(bv < 0.0 ? 0.0 : bv);
    const double f0 = fabs(M.A[M.at(p, from)]);
    const unsigned long long hit = __ballot(bv == bm);
    int t = from;
    if (f0 == f0 && hit != 0)
        t = (hit & (hit - 1)) == 0 ? __builtin_amdgcn_readlane(bi, __builtin_ctzll(hit))
                                   : __builtin_amdgcn_readfirstlane(wave_min_int(bv == bm ? bi : INT_MAX));
    const double app = M.A[p + p * M.ld], apt = M.A[M.at(p, t)], att = M.A[t + t * M.ld];
    // max over the line without t: a lane whose own best is t gives its others
    const double maxp = wave_max_abs(max_abs(oth, (bi == t || bv < 0.0) ? 0.0 : bv));
    const double maxt = tpp_line_max(M, t, from, p);
    *tout = t;
    if (tpp_test_2x2(att, apt, app, maxt, maxp, u, small)) return TPP_2X2;
    return (fabs(app) >= u * fmax(maxp, fabs(apt))) ? TPP_1X1 : TPP_NONE;
}

// Symmetric exchange of lines i < j (all threads; the pairs of line q are disjoint).
template <int NT, class P>
__device__ __forceinline__ void tpp_swap(const TppMat<P> &M, int *lperm, int i, int j) {
    if (i == j) return;
    if (i > j) { const int t = i; i = j; j = t; }
    for (int q0 = threadIdx.x; q0 < M.m; q0 += NT * TPP_B) {
        size_t a1[TPP_B], a2[TPP_B];
        double x1[TPP_B], x2[TPP_B];
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) {
            const int q = q0 + NT * t;
            const bool ok = q < M.m && q != i && q != j;
            a1[t] = ok ? M.at(i, q) : i + i * M.ld;
            a2[t] = ok ? M.at(j, q) : i + i * M.ld;
            x1[t] = M.A[a1[t]];
            x2[t] = M.A[a2[t]];
        }
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) {
            const int q = q0 + NT * t;
            if (q < M.m && q != i && q != j) { M.A[a1[t]] = x2[t]; M.A[a2[t]] = x1[t]; }
        }
    }
    if (threadIdx.x == 0) {
        const double t = M.A[i + i * M.ld]; M.A[i + i * M.ld] = M.A[j + j * M.ld]; M.A[j + j * M.ld] = t;
        const int pt = lperm[i]; lperm[i] = lperm[j]; lperm[j] = pt;
    }
    __syncthreads();
}

// Elimination of the 1x1 at ne (two = false) or the 2x2 at ne, ne + 1: the columns scaled to L, then
// the fully-summed columns updated, TJ per wavefront and pass.  LB: the new columns of L are also
// kept in lb (LDS, 2 m doubles) and read from there, so that a pass over a front in memory waits
// for its own entries only.  Returns the thread's largest |l|.
template <int NT, int TJ, int RB, bool LB, class P>
__device__ __forceinline__ double tpp_apply(const TppMat<P> &M, int ne, bool two, double *lb) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    P A = M.A;
    const size_t ld = M.ld;
    const int nx = ne + (two ? 2 : 1);
    const double a11 = A[ne + ne * ld];
    double a21 = 0.0, a22 = 0.0;
    if (two) { a21 = A[(ne + 1) + ne * ld]; a22 = A[(ne + 1) + (ne + 1) * ld]; }
    const double inv = 1.0 / (two ? a11 * a22 - a21 * a21 : a11);
    double ml = 0.0;
    for (int i0 = nx + tid; i0 < M.m; i0 += NT * TPP_B) {
        double v1[TPP_B], v2[TPP_B];
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) {
            const int i = min(i0 + NT * t, M.m - 1);
            v1[t] = A[i + ne * ld];
            v2[t] = two ? A[i + (ne + 1) * ld] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < TPP_B; ++t) {
            const int i = i0 + NT * t;
            if (i >= M.m) continue;
            if (two) {
                const double l1 = (v1[t] * a22 - v2[t] * a21) * inv;
                const double l2 = (v2[t] * a11 - v1[t] * a21) * inv;
                A[i + ne * ld] = l1;
                A[i + (ne + 1) * ld] = l2;
                if (LB) { lb[i] = l1; lb[M.m + i] = l2; }
                ml = max_abs(max_abs(ml, l1), l2);
            } else {
                const double l = v1[t] * inv;
                A[i + ne * ld] = l;
                if (LB) lb[i] = l;
                ml = max_abs(ml, l);
            }
        }
    }
    __syncthreads();
    for (int j0 = nx + wv * TJ; j0 < M.n; j0 += (NT / 64) * TJ) {
        double w1[TJ], w2[TJ];
#pragma unroll
        for (int q = 0; q < TJ; ++q) {
            const int j = min(j0 + q, M.n - 1);
            const double lj1 = LB ? lb[j] : A[j + ne * ld];
            if (two) {
                const double lj2 = LB ? lb[M.m + j] : A[j + (ne + 1) * ld];
                w1[q] = lj1 * a11 + lj2 * a21;
                w2[q] = lj1 * a21 + lj2 * a22;
            } else {
                w1[q] = lj1 * a11;
                w2[q] = 0.0;
            }
        }
        // RB rows per lane at a time, every load of a batch before its stores
        for (int i0 = j0 + lane; i0 < M.m; i0 += 64 * RB) {
            double c[TJ][RB], l1[RB], l2[RB];
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                const int i = min(i0 + 64 * r, M.m - 1);
                l1[r] = LB ? lb[i] : A[i + ne * ld];
                l2[r] = !two ? 0.0 : LB ? lb[M.m + i] : A[i + (ne + 1) * ld];
#pragma unroll
                for (int q = 0; q < TJ; ++q) c[q][r] = A[i + min(j0 + q, M.n - 1) * ld];
            }
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int q = 0; q < TJ; ++q) {
                    const int i = i0 + 64 * r;
                    const double x = two ? l1[r] * w1[q] + l2[r] * w2[q] : l1[r] * w1[q];
                    if (j0 + q < M.n && i >= j0 + q && i < M.m) A[i + (j0 + q) * ld] = c[q][r] - x;
                }
        }
    }
    __syncthreads();
    if (two) {
        if (tid == 0) A[(ne + 1) + ne * ld] = 0.0;
        __syncthreads();
    }
    return ml;
}

// LDS of a staged front: its trapezoid's columns with an odd leading dimension (rows and columns
// are read without bank conflicts), and the row order.
__host__ __device__ __forceinline__ size_t tpp_lds_bytes(int m, int n) {
    return ((size_t)(m | 1) * n * 8 + (size_t)n * 4 + 15) / 16 * 16;
}
constexpr size_t TPP_LDS_MAX = 158 * 1024;  // beside the workgroup's static LDS
constexpr size_t TPP_LDS_SMALL = 38 * 1024;  // four workgroups per CU

// The launches of a level's TPP fronts.
//  * TPP_SMALL: four wavefronts per front, staged, at least four fronts to a CU.
//  * TPP_WAVE, for more than TPP_WAVE_MIN fronts of at most a row per lane: one wavefront each, sixteen
//    to a CU.  Four scan a line no sooner, and their idle lanes and barriers take the place of three other
//    fronts.  Refactorization of independent systems, one / four wavefronts, ms: 24 x 24, 500 of
//    them 0.14 / 0.12, 1000 0.17 / 0.18, 2000 0.21 / 0.27, 20000 1.10 / 2.02; 8 x 8, 1000 0.08 / 0.10,
//    2000 0.11 / 0.14, 20000 0.54 / 0.89.
//  * TPP_MID, for more than TPP_MID_MIN fronts of which only one fits on a CU: in place on two wavefronts
//    until the rest is small, four to a CU.  Up to that number staging them whole is the shorter
//    chain, and so it is where two fit.  In parts / whole, ms: 104 x 104, 512 of them 0.94 / 0.92, 700
//    1.05 / 1.28, 3000 3.42 / 4.93; 120 x 120, 200 0.92 / 0.59, 512 1.17 / 1.08, 700 1.32 / 1.52, 3000 4.29 /
//    5.80; 140 x 140, 512 1.56 / 1.33, 700 1.74 / 1.90, 3000 5.93 / 7.42; 100 x 100, 700 0.98 / 0.94, 6000
//    6.14 / 6.03; past the LDS (160 x 160) 700 2.63 / 2.46, 6000 18.7 / 18.7.
//  * TPP_WIDE: four wavefronts, staged whole or in place throughout.
enum TppClass { TPP_WAVE = 0, TPP_SMALL = 1, TPP_MID = 2, TPP_WIDE = 3 };
constexpr int TPP_WAVE_MIN = 1024, TPP_MID_MIN = 512;
constexpr size_t TPP_LDS_WAVE = 10 * 1024, TPP_LDS_HALF = 79 * 1024;

// Threshold partial pivoting of a front's columns from c0 on, until what is left fits in lds bytes
// (0: to the end).  Returns the columns eliminated; the row order in lperm.
template <int NT, int TJ, int RB, bool LB, class P>
__device__ __forceinline__ int tpp_run(const TppMat<P> &M, FrontDev &F, int c0, int *lperm, double u, double small,
                                       unsigned lds, double *lb) {
    constexpr int NW = NT / 64;
    __shared__ int s_code[NW], s_t[NW], s_ok;
    __shared__ double s_ml[NW];
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = M.n;
    int nelim = 0, n1 = 0, n2 = 0;
    double ml = 0.0;
    for (int i = tid; i < n; i += NT) lperm[i] = i;
    __syncthreads();
    auto set1 = [&](int col, double v) {
        if (tid == 0) { gbl(F.dkind)[c0 + col] = 1; gbl(F.ddiag)[c0 + col] = v; gbl(F.doff)[c0 + col] = 0.0; }
    };
    while (nelim < n && !(lds && tpp_lds_bytes(M.m - nelim, n - nelim) <= lds)) {
        // rounds of candidates: in the first, wavefront 0 looks at column nelim itself
        int code = TPP_NONE, p = nelim, t = nelim;
        bool last_ok = false;
        int base = nelim;
        for (;;) {
            const int c = base + wv;
            int cd = TPP_NONE, ct = 0;
            if (c == nelim) {
                bool big;
                const double mp = tpp_line_max(M, nelim, nelim, -1, small, &big);
                const double d = fabs(M.A[nelim + nelim * M.ld]);
                if (!big && !(d >= small)) cd = TPP_ZERO;
                if ((tid & 63) == 0) s_ok = d >= u * mp;
            } else if (c < n) {
                cd = tpp_candidate(M, c, nelim, u, small, &ct);
            }
            if ((tid & 63) == 0) { s_code[wv] = cd; s_t[wv] = ct; }
            __syncthreads();
#pragma unroll
            for (int w = NW - 1; w >= 0; --w)
                if (s_code[w] != TPP_NONE) { code = s_code[w]; p = base + w; t = s_t[w]; }
            last_ok = s_ok != 0;
            __syncthreads();
            base += NW;
            if (code != TPP_NONE || base >= n) break;
        }
        code = __builtin_amdgcn_readfirstlane(code);
        p = __builtin_amdgcn_readfirstlane(p);
        t = __builtin_amdgcn_readfirstlane(t);
        if (code == TPP_ZERO) {
            tpp_swap<NT>(M, lperm, p, nelim);
            set1(nelim, 0.0);
            ++n1;
            for (int r = nelim + 1 + tid; r < M.m; r += NT) M.A[r + nelim * M.ld] = 0.0;
            __syncthreads();
            nelim += 1;
        } else if (code == TPP_2X2) {
            tpp_swap<NT>(M, lperm, t, nelim);
            const int np = (p == nelim) ? t : p;
            tpp_swap<NT>(M, lperm, np, nelim + 1);
            if (tid == 0) {
                gbl(F.dkind)[c0 + nelim] = 2; gbl(F.dkind)[c0 + nelim + 1] = 3;
                gbl(F.ddiag)[c0 + nelim] = M.A[nelim + nelim * M.ld];
                gbl(F.ddiag)[c0 + nelim + 1] = M.A[(nelim + 1) + (nelim + 1) * M.ld];
                gbl(F.doff)[c0 + nelim] = M.A[(nelim + 1) + nelim * M.ld]; gbl(F.doff)[c0 + nelim + 1] = 0.0;
            }
            ml = max_abs(ml, tpp_apply<NT, TJ, RB, LB>(M, nelim, true, lb));
            ++n2;
            nelim += 2;
        } else {
            if (code == TPP_NONE) {  // the 1x1 test of column nelim itself comes last
                if (!last_ok) break;
                p = nelim;
            }
            tpp_swap<NT>(M, lperm, p, nelim);
            set1(nelim, M.A[nelim + nelim * M.ld]);
            ml = max_abs(ml, tpp_apply<NT, TJ, RB, LB>(M, nelim, false, lb));
            ++n1;
            nelim += 1;
        }
    }
    ml = wave_max_abs(ml);
    if ((tid & 63) == 0) s_ml[wv] = ml;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < NW; ++w) ml = max_abs(ml, s_ml[w]);
        F.ne = c0 + nelim;
        F.n1 += n1;
        F.n2 += n2;
        atomic_max_nonneg(&F.max_l_bits, ml);
    }
    return nelim;
}

// A front's columns from c0 on by one workgroup.  A pivot step is a serial chain of scans, so its
// memory round trips decide: the columns still to eliminate are staged in LDS where they fit (lds
// bytes).  PARTS: wider remainders are worked on in place until the rest fits, the step's new columns
// of L kept in LDS (without it a wide front is worked on in place throughout, the kernel keeps to
// few registers).  Rows of earlier columns follow the row order at the end of either part.
// KKT of side 16 (fronts up to 131 x 131): about 5 us a step, 26 us with every scan through L2 and a
// workgroup reduction of its own.  422 left-over columns at the root of KKT 45: 5.3 ms in place
// throughout on 1024 threads, 3.8 so on 512 (24 -> 15 us a step in memory, 4.7 staged).
template <int NT, int TJ, bool PARTS>
__device__ __forceinline__ void tpp_front(FrontDev &F, int c0, double u, double small, unsigned lds, double *dyn) {
    const size_t lda = F.m;
    const int tid = threadIdx.x;
    for (bool more = c0 < F.k; more;) {
        const int n = F.k - c0, m = F.m - c0;
        gdouble *G = gbl(F.F) + c0 + c0 * lda;
        int *lperm;
        int nelim = 0;
        more = false;
        if (tpp_lds_bytes(m, n) <= lds) {
            const size_t ld = m | 1;
            lperm = (int *)(dyn + ld * n);
            for (int j0 = tid >> 6; j0 < n; j0 += NT / 64 * 4)
                for (int i = (tid & 63); i < m; i += 64) {
                    double v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = G[i + (size_t)min(j0 + q * (NT / 64), n - 1) * lda];
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (j0 + q * (NT / 64) < n) dyn[i + (j0 + q * (NT / 64)) * ld] = v[q];
                }
            __syncthreads();
            tpp_run<NT, TJ, 2, false>(TppMat<double *>{dyn, ld, m, n}, F, c0, lperm, u, small, 0, nullptr);
            for (int j = tid >> 6; j < n; j += NT / 64)
                for (int i = j + (tid & 63); i < m; i += 64) G[i + (size_t)j * lda] = dyn[i + j * ld];
        } else {
            lperm = F.sidx + c0;  // (written by k_collect after the factorization)
            const TppMat<gdouble *> M{G, lda, m, n};
            if (PARTS && (size_t)m * 16 <= lds) {
                nelim = tpp_run<NT, TJ, 4, true>(M, F, c0, lperm, u, small, lds, dyn);
                more = nelim < n && tpp_lds_bytes(m - nelim, n - nelim) <= lds;
            } else {
                tpp_run<NT, TJ, 4, false>(M, F, c0, lperm, u, small, 0, nullptr);
            }
        }
        __syncthreads();
        // perm and the earlier columns' rows [c0, c0 + n) in the new order, columns dealt to the wavefronts
        // (one register per lane and 64 rows; every load of a column before its stores)
        gint *perm = gbl(F.perm) + c0;
        constexpr int RB = 16;
        if (n <= 64 * RB) {
            for (int q = (tid >> 6) - 1; q < c0; q += NT / 64) {
                gdouble *col = gbl(F.F) + c0 + (size_t)max(q, 0) * lda;
                double v[RB];
                int pv[RB];
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    const int i = (tid & 63) + 64 * r;
                    if (i >= n) continue;
                    if (q < 0) pv[r] = perm[lperm[i]];
                    else v[r] = col[lperm[i]];
                }
                __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    const int i = (tid & 63) + 64 * r;
                    if (i >= n) continue;
                    if (q < 0) perm[i] = pv[r];
                    else col[i] = v[r];
                }
            }
        } else {
            // more columns left over: one column per thread, cycle by cycle (from each cycle's smallest row)
            for (int q = tid - 1; q < c0; q += NT) {
                gdouble *col = gbl(F.F) + c0 + (size_t)max(q, 0) * lda;
                for (int i = 0; i < n; ++i) {
                    int a = lperm[i];
                    while (a > i) a = lperm[a];
                    if (a < i || lperm[i] == i) continue;
                    const double v = col[i];
                    const int pv = q < 0 ? perm[i] : 0;
                    a = i;
                    for (int b; (b = lperm[a]) != i; a = b) {
                        if (q < 0) perm[a] = perm[b];
                        else col[a] = col[b];
                    }
                    if (q < 0) perm[a] = pv;
                    else col[a] = v;
                }
            }
        }
        c0 += nelim;
        __syncthreads();
    }
}

// Whole fronts, one workgroup each.
template <int NT, int TJ, bool PARTS>
__global__ __launch_bounds__(NT) void k_tpp(FrontDev *__restrict__ fr, const int *__restrict__ flist, double u,
                                            double small, unsigned lds) {
    extern __shared__ __align__(16) double dyn[];
    tpp_front<NT, TJ, PARTS>(fr[flist[blockIdx.x]], 0, u, small, lds, dyn);
}

// The columns APTP left over, of the fronts that have some.  Its LDS lets one workgroup onto a CU, so
// TPP_LEFT_WG of them take the fronts of the list in turn: a workgroup for every front of the level
// cost 60 us at 4000 fronts of order 40 (280 at order 180), most of them without such a column.
constexpr int TPP_LEFT_WG = 256;
template <int NT, int TJ>
__global__ __launch_bounds__(NT) void k_tpp_left(FrontDev *__restrict__ fr, const int *__restrict__ left, double u,
                                                 double small, unsigned lds) {
    extern __shared__ __align__(16) double dyn[];
    const int n = left[0];
    for (int f = blockIdx.x; f < n; f += gridDim.x) {
        FrontDev &F = fr[left[1 + f]];
        tpp_front<NT, TJ, true>(F, F.ne, u, small, lds, dyn);
    }
}

// ===========================================================================
// Schur updates on FP64 MFMA: C -= W L_c^T on the lower part, with W = L_r D formed once per
// update by k_form_ld.
//   mode 0 (contribution, compute_contribution_gemm factor.rs:1590-1652):
//           rows/cols [k, m), K = ne columns from 0.
//   mode 1 (outer-block update of the deferred trailing columns):
//           rows [obe, m), cols [obe, k), K = columns eliminated in the outer block.
// ===========================================================================
typedef double d4 __attribute__((ext_vector_type(4)));

struct UpdGeom {
    int r0, nr, nc, kc0, K;
};

__device__ __forceinline__ UpdGeom upd_geom(const FrontDev &F, const AptpState *st, int aux, int mode) {
    UpdGeom g;
    if (mode == 0) {
        g.r0 = F.k; g.nr = F.m - F.k; g.nc = g.nr; g.kc0 = 0; g.K = F.ne;
    } else {
        const AptpState &S = st[aux];
        g.r0 = S.ob_start + S.ob_cols; g.nr = F.m - g.r0; g.nc = F.k - g.r0; g.kc0 = S.ob_start;
        g.K = S.kpos - S.ob_start;
    }
    return g;
}

constexpr int FC = 32;  // columns per k_form_ld work item

// W[r, c] = (L D)[r0 + r, kc0 + c] (compute_ld_into, factor.rs:1536-1563), column-major with
// leading dimension nr.  Work item (front, aux, 256 rows, FC columns).  For an FP32 front
// (FRONT_W32) the workspace holds W and a copy of L[r0 + r, kc0 + c] as FP32, each nr x K with
// leading dimension nr (together the bytes of the FP64 W): the rounding k_schur<1> applies to its
// operands, done once per front instead of once per tile, and half the operand bytes per tile.
// snap (mode 1, may be null): the first item of each front copies the front's APTP state there,
// for an outer update that runs after the state has moved on to the next outer block.
__global__ __launch_bounds__(256) void k_form_ld(const FrontDev *__restrict__ fr,
                                                 const AptpState *__restrict__ st,
                                                 const int4 *__restrict__ items, int mode,
                                                 double *const *__restrict__ wp,
                                                 AptpState *__restrict__ snap) {
    const int4 it = items[blockIdx.x];
    const FrontDev &F = fr[it.x];
    if (snap && it.z == 0 && it.w == 0) {
        const int *src = (const int *)&st[it.y];
        int *dst = (int *)&snap[it.y];
        for (int i = threadIdx.x; i < (int)(sizeof(AptpState) / sizeof(int)); i += blockDim.x) dst[i] = src[i];
    }
    const UpdGeom g = upd_geom(F, st, it.y, mode);
    if (g.K <= 0 || g.nr <= 0) return;
    const int c0 = it.w * FC;
    if (c0 >= g.K) return;
    const int cn = min(FC, g.K - c0);
    __shared__ int sk[FC + 2];
    __shared__ double sd[FC + 2], so[FC + 2];
    const int tid = threadIdx.x;
    if (tid < FC + 2) {
        const int c = c0 - 1 + tid;
        const bool in = c >= 0 && c < g.K;
        sk[tid] = in ? gbl(F.dkind)[g.kc0 + c] : 0;
        sd[tid] = in ? gbl(F.ddiag)[g.kc0 + c] : 0.0;
        so[tid] = in ? gbl(F.doff)[g.kc0 + c] : 0.0;
    }
    __syncthreads();
    const int r = it.z * 256 + tid;
    if (r >= g.nr) return;
    const size_t lda = F.m;
    const gdouble *row = gbl(F.F) + (g.r0 + r);
    double lv[FC + 2];
#pragma unroll
    for (int u = 0; u < FC + 2; ++u) {
        const int c = c0 - 1 + u;
        lv[u] = (c >= 0 && c < g.K) ? row[(size_t)(g.kc0 + c) * lda] : 0.0;
    }
    const bool w32 = (F.flags & FRONT_W32) != 0;
    gdouble *W = gbl(wp[it.y]) + r;
    __attribute__((address_space(1))) float *W32 = (__attribute__((address_space(1))) float *)gbl(wp[it.y]) + r;
    __attribute__((address_space(1))) float *L32 = W32 + (size_t)g.nr * g.K;
#pragma unroll
    for (int u = 1; u <= FC; ++u) {
        if (u - 1 < cn) {
            const int kind = sk[u];
            double v = 0.0;
            if (kind == 1) v = lv[u] * sd[u];
            else if (kind == 2) v = lv[u] * sd[u] + lv[u + 1] * so[u];
            else if (kind == 3) v = lv[u - 1] * so[u - 1] + lv[u] * sd[u];
            const size_t o = (size_t)(c0 + u - 1) * g.nr;
            if (w32) {
                W32[o] = (float)v;
                L32[o] = (float)lv[u];
            } else {
                W[o] = v;
            }
        }
    }
}

typedef float f4 __attribute__((ext_vector_type(4)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// Workgroup -> tile-list index.  Consecutive workgroups are dispatched round-robin over the 8
// XCDs (workgroup bid runs on XCD bid & 7).
//  * contiguous (contribution updates, every listed tile active): each XCD takes one contiguous
//    run of the list, so tiles of a row block share W rows in its L2;
//  * spread (outer-block updates): the list is planned for the largest trailing block, and only a
//    prefix of each front's tiles is active once earlier outer blocks have been eliminated; runs
//    of TILE_RUN consecutive tiles go to successive XCDs, so every prefix is spread over all of
//    them.  The grid is rounded up to a multiple of 8 * TILE_RUN; indices >= ntiles are idle.
constexpr unsigned TILE_RUN = 2;
__host__ __device__ constexpr unsigned spread_grid(size_t ntiles) {
    return (unsigned)((ntiles + 8 * TILE_RUN - 1) / (8 * TILE_RUN) * (8 * TILE_RUN));
}
__device__ __forceinline__ unsigned tile_index(unsigned bid, unsigned nbk, bool spread) {
    const unsigned xcd = bid & 7, s = bid >> 3;
    if (spread) return ((s / TILE_RUN) * 8 + xcd) * TILE_RUN + s % TILE_RUN;
    const unsigned qn = nbk >> 3, rem = nbk & 7;
    return xcd * qn + min(xcd, rem) + s;
}

// FP64 -> BF16 bits, round to nearest even (through FP32, itself rounded to nearest)
__device__ __forceinline__ unsigned short to_bf16(double x) {
    unsigned u = __float_as_uint((float)x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

// C -= W L_c^T: 128 x 128 output tile per workgroup (4 wavefronts x 64 x 64 = 4 x 4 MFMA
// 16x16 blocks), K in chunks of SKC through LDS with the next chunk prefetched into registers
// (a chunk's MFMA work outlasts the global-load latency).  The operands enter the MFMA as
// (L_c, W), so a lane's four results lie in one row of C.
//   PREC 0: FP64 operands, v_mfma_f64_16x16x4f64;
//   PREC 1: operands rounded to FP32, v_mfma_f32_16x16x4f32, FP32 accumulation;
//   PREC 2: operands rounded to BF16, v_mfma_f32_16x16x32_bf16, FP32 accumulation.
// The product is subtracted from the FP64 C in every case.
constexpr int SKC = 32;

// Two workgroups per CU for FP64 and BF16, three for FP32 (registers fit 256 resp. 168 per lane);
// FP64 and FP32 take K in chunks of 16 so that their double-buffered operand tiles fit that many
// times in the LDS.  TILE = 64 (FP64 / FP32 only): 64 x 64 output tiles, each wavefront a 32 x 32
// quarter, for the thin updates on the critical path (four times the workgroups of 128 x 128
// tiles over the same columns); every entry is summed in the same order either way.
template <int PREC, int TILE = 128>
__global__ __launch_bounds__(256, PREC == 1 ? 3 : 2) void k_schur(const FrontDev *__restrict__ fr,
                                               const AptpState *__restrict__ st,
                                               const TileItem *__restrict__ tiles, int mode,
                                               double *const *__restrict__ wp, unsigned ntiles) {
    static_assert(TILE == 128 || (TILE == 64 && PREC != 2), "tile: 128, or 64 for FP64 / FP32");
    constexpr int KCH = (PREC == 2) ? SKC : 16;  // K per chunk (the LDS of two FP64 / three FP32 workgroups per CU)
    constexpr int NB = TILE / 32;                 // 16 x 16 MFMA blocks per wavefront and dimension
    constexpr int WS = TILE / 2;                  // a wavefront's sub-tile
    constexpr int KS = 256 / TILE;                // k slices of a chunk's operand loads
    constexpr int P64 = TILE + 8, P32 = TILE + 16;  // LDS row pitches (FP64, FP32)
    const unsigned ti_ = tile_index(blockIdx.x, gridDim.x, mode == 1);
    if (ti_ >= ntiles) return;
    const TileItem t = tiles[ti_];
    const FrontDev &F = fr[t.front];
    const UpdGeom g = upd_geom(F, st, t.aux, mode);
    const int K = g.K, nr = g.nr, nc = g.nc, r0 = g.r0;
    if (K <= 0 || nr <= 0 || nc <= 0) return;
    const int bi = t.ti * TILE, bj = t.tj * TILE;
    if (bi >= nr || bj >= nc || bi + TILE - 1 < bj) return;
    const size_t lda = F.m;
    gdouble *A = gbl(F.F);
    // LDS operand tiles: [k][row] for FP64/FP32, [row][k] for BF16 (four consecutive k per lane)
    // two chunk buffers: a chunk is staged while the previous one feeds the MFMAs (one barrier
    // per chunk)
    constexpr int LDS_BYTES = (PREC == 0) ? 2 * KCH * P64 * 8 : (PREC == 1) ? 2 * KCH * P32 * 4
                                                                             : 2 * 128 * (KCH + 8) * 2;
    __shared__ __align__(16) char lds2[2 * LDS_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wr = wv >> 1, wc = wv & 1;
    // a wavefront whose sub-tile lies strictly above the diagonal only helps staging
    const bool busy = bi + wr * WS + WS - 1 >= bj + wc * WS;
    const int lr = tid % TILE, ko = tid / TILE;
    const bool arow = bi + lr < nr, brow = bj + lr < nc;
    // operand loads through buffer resources based at the chunk's first column: an entry outside
    // the tile or beyond K gets an out-of-range offset and loads as zero, with no branch and no
    // select, so the waits count the loads of the chunk in flight exactly
    // FP32: W and L come as FP32 pairs from the workspace (k_form_ld, FRONT_W32); otherwise W
    // (FP64) from the workspace and L from the front
    typedef typename std::conditional<PREC == 1, float, double>::type op_t;
    const double *Wb = wp[t.aux] + bi;
    const double *Lb = F.F + (r0 + bj) + (size_t)g.kc0 * lda;
    const float *W32 = (const float *)wp[t.aux] + bi;
    const float *L32 = (const float *)wp[t.aux] + (size_t)nr * K + bj;
    auto load_chunk = [&](op_t *ra, op_t *rb, int kc) {
        if constexpr (PREC == 1) {
            const __amdgpu_buffer_rsrc_t rw = buf_rsrc(W32 + (size_t)kc * nr);
            const __amdgpu_buffer_rsrc_t rl = buf_rsrc(L32 + (size_t)kc * nr);
#pragma unroll
            for (int u = 0; u < KCH / KS; ++u) {
                const int cc = ko + KS * u, c = kc + cc;
                ra[u] = buf_load_f32(rw, (arow && c < K) ? (unsigned)(lr + cc * nr) * 4u : BUF_OOB);
                rb[u] = buf_load_f32(rl, (brow && c < K) ? (unsigned)(lr + cc * nr) * 4u : BUF_OOB);
            }
        } else {
            const __amdgpu_buffer_rsrc_t rw = buf_rsrc(Wb + (size_t)kc * nr);
            const __amdgpu_buffer_rsrc_t rl = buf_rsrc(Lb + (size_t)kc * lda);
#pragma unroll
            for (int u = 0; u < KCH / KS; ++u) {
                const int cc = ko + KS * u, c = kc + cc;
                ra[u] = buf_load_f64(rw, (arow && c < K) ? (unsigned)(lr + cc * nr) * 8u : BUF_OOB);
                rb[u] = buf_load_f64(rl, (brow && c < K) ? (unsigned)(lr + cc * (int)lda) * 8u : BUF_OOB);
            }
        }
    };
    constexpr int NU = KCH / KS;  // k values per thread and operand in one chunk
    typedef typename std::conditional<PREC == 0, d4, f4>::type acc_t;
    acc_t acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    // a chunk's operands in registers into its LDS buffer
    auto stage = [&](const op_t *ra, const op_t *rb, char *lds) {
        if constexpr (PREC == 0) {
            double (*As)[P64] = (double (*)[P64])lds;
            double (*Bs)[P64] = (double (*)[P64])(lds + KCH * P64 * 8);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                As[ko + KS * u][lr] = ra[u];
                Bs[ko + KS * u][lr] = rb[u];
            }
        } else if constexpr (PREC == 1) {
            float (*As)[P32] = (float (*)[P32])lds;
            float (*Bs)[P32] = (float (*)[P32])(lds + KCH * P32 * 4);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                As[ko + KS * u][lr] = (float)ra[u];
                Bs[ko + KS * u][lr] = (float)rb[u];
            }
        } else {
            unsigned short (*As)[KCH + 8] = (unsigned short (*)[KCH + 8])lds;
            unsigned short (*Bs)[KCH + 8] = (unsigned short (*)[KCH + 8])(lds + 128 * (KCH + 8) * 2);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                As[lr][ko + 2 * u] = to_bf16(ra[u]);
                Bs[lr][ko + 2 * u] = to_bf16(rb[u]);
            }
        }
    };
    // the MFMAs of one staged chunk
    auto compute = [&](char *lds) {
        if (busy) {
            if constexpr (PREC == 0) {
                double (*As)[P64] = (double (*)[P64])lds;
                double (*Bs)[P64] = (double (*)[P64])(lds + KCH * P64 * 8);
#pragma unroll
                for (int kk = 0; kk < KCH; kk += 4) {
                    const int kr = kk + (lane >> 4);
                    double a[NB], b[NB];
#pragma unroll
                    for (int i = 0; i < NB; ++i) a[i] = As[kr][wr * WS + i * 16 + (lane & 15)];
#pragma unroll
                    for (int j = 0; j < NB; ++j) b[j] = Bs[kr][wc * WS + j * 16 + (lane & 15)];
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j], a[i], acc[i][j], 0, 0, 0);
                }
            } else if constexpr (PREC == 1) {
                float (*As)[P32] = (float (*)[P32])lds;
                float (*Bs)[P32] = (float (*)[P32])(lds + KCH * P32 * 4);
#pragma unroll
                for (int kk = 0; kk < KCH; kk += 4) {
                    const int kr = kk + (lane >> 4);
                    float a[NB], b[NB];
#pragma unroll
                    for (int i = 0; i < NB; ++i) a[i] = As[kr][wr * WS + i * 16 + (lane & 15)];
#pragma unroll
                    for (int j = 0; j < NB; ++j) b[j] = Bs[kr][wc * WS + j * 16 + (lane & 15)];
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], a[i], acc[i][j], 0, 0, 0);
                }
            } else {
                unsigned short (*As)[KCH + 8] = (unsigned short (*)[KCH + 8])lds;
                unsigned short (*Bs)[KCH + 8] = (unsigned short (*)[KCH + 8])(lds + 128 * (KCH + 8) * 2);
                // v_mfma_f32_16x16x32_bf16: lane l holds eight consecutive k, 8 (l / 16) .. + 7,
                // of row / column l % 16
#pragma unroll
                for (int kk = 0; kk < KCH; kk += 32) {
                    const int k8 = kk + 8 * (lane >> 4);
                    bf8 a[4], b[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) a[i] = *(const bf8 *)&As[wr * 64 + i * 16 + (lane & 15)][k8];
#pragma unroll
                    for (int j = 0; j < 4; ++j) b[j] = *(const bf8 *)&Bs[wc * 64 + j * 16 + (lane & 15)][k8];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
                }
            }
        }
    };
    // the next chunk's operands are loaded while the current one feeds the MFMAs
    op_t ra[NU], rb[NU];
    load_chunk(ra, rb, 0);
    for (int kc = 0, buf = 0; kc < K; kc += KCH, buf ^= 1) {
        char *lds = lds2 + buf * LDS_BYTES;
        stage(ra, rb, lds);
        __syncthreads();
        if (kc + KCH < K) load_chunk(ra, rb, kc + KCH);
        compute(lds);
    }
    if (!busy) return;
    // result layouts, (L_c, W) product: v_mfma_f64_16x16x4f64 lane l element q holds D row
    // (l/16) + 4q, column l%16; the FP32-accumulating 16x16 MFMAs hold D row 4(l/16) + q.
    // D row = C column, D column = C row.  C's entries are loaded before any is stored, half of
    // the tile at a time (a store may alias a later load, so interleaved read-modify-writes would
    // take one memory round trip each); entries outside the lower tile load as zero and are not
    // stored.
    const int rl0 = bi + wr * WS + (lane & 15);
    const __amdgpu_buffer_rsrc_t rc = buf_rsrc(F.F + (r0 + bi) + (size_t)(r0 + bj) * lda);  // tile origin
    constexpr int NH = (NB + 1) / 2;  // row blocks per half
#pragma unroll
    for (int h = 0; h < NB / NH; ++h) {
        double cv[NH][NB][4];
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int rl = rl0 + (NH * h + i) * 16;
                    const int dr = (PREC == 0) ? (lane >> 4) + 4 * q : 4 * (lane >> 4) + q;
                    const int cl = bj + wc * WS + j * 16 + dr;
                    const bool ok = rl < nr && cl < nc && rl >= cl;
                    const unsigned off = (unsigned)((rl - bi) + (size_t)(cl - bj) * lda) * 8u;
                    cv[i][j][q] = buf_load_f64(rc, ok ? off : BUF_OOB);
                }
#pragma unroll
        for (int i = 0; i < NH; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int rl = rl0 + (NH * h + i) * 16;
                    const int dr = (PREC == 0) ? (lane >> 4) + 4 * q : 4 * (lane >> 4) + q;
                    const int cl = bj + wc * WS + j * 16 + dr;
                    if (rl < nr && cl < nc && rl >= cl)
                        A[(r0 + rl) + (size_t)(r0 + cl) * lda] = cv[i][j][q] - (double)acc[NH * h + i][j][q];
                }
    }
}

// C -= W L_c^T in the oracle's summation order (gemm_sub_wlt): every entry accumulates
// W[i,c] * L[j,c] over c ascending from zero, multiply and add rounded separately (this file
// is compiled without FMA contraction), and is subtracted once.  128 x 128 tile per workgroup,
// each thread 8 rows x 8 columns; K staged through LDS in chunks of SKC.
__global__ __launch_bounds__(256) void k_schur_exact(const FrontDev *__restrict__ fr,
                                                     const AptpState *__restrict__ st,
                                                     const TileItem *__restrict__ tiles, int mode,
                                                     double *const *__restrict__ wp, unsigned ntiles) {
    const unsigned ti_ = tile_index(blockIdx.x, gridDim.x, mode == 1);
    if (ti_ >= ntiles) return;
    const TileItem t = tiles[ti_];
    const FrontDev &F = fr[t.front];
    const UpdGeom g = upd_geom(F, st, t.aux, mode);
    const int K = g.K, nr = g.nr, nc = g.nc, r0 = g.r0;
    if (K <= 0 || nr <= 0 || nc <= 0) return;
    const int bi = t.ti * 128, bj = t.tj * 128;
    if (bi >= nr || bj >= nc || bi + 127 < bj) return;
    const size_t lda = F.m;
    gdouble *A = gbl(F.F);
    __shared__ double As[SKC][132];
    __shared__ double Bs[SKC][132];
    const int tid = threadIdx.x;
    const int tr = tid & 15, tc = tid >> 4;  // rows tr + 16a, columns tc + 16b
    const int lr = tid & 127, ko = tid >> 7;
    const bool arow = bi + lr < nr, brow = bj + lr < nc;
    const gdouble *Wp = gbl(wp[t.aux]) + bi + lr;
    const gdouble *Lp = A + (r0 + bj + lr) + (size_t)g.kc0 * lda;
    auto load_chunk = [&](double *ra, double *rb, int kc) {
#pragma unroll
        for (int u = 0; u < SKC / 2; ++u) {
            const int c = kc + ko + 2 * u;
            ra[u] = (arow && c < K) ? Wp[(size_t)c * nr] : 0.0;
            rb[u] = (brow && c < K) ? Lp[(size_t)c * lda] : 0.0;
        }
    };
    constexpr int NU = SKC / 2;
    double ra[NU], rb[NU];
    load_chunk(ra, rb, 0);
    double acc[8][8];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[a][b] = 0.0;
    for (int kc = 0; kc < K; kc += SKC) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            As[ko + 2 * u][lr] = ra[u];
            Bs[ko + 2 * u][lr] = rb[u];
        }
        __syncthreads();
        if (kc + SKC < K) load_chunk(ra, rb, kc + SKC);
        const int kn = min(SKC, K - kc);  // products beyond K are not added
        for (int kk = 0; kk < kn; ++kk) {
            double av[8], bv[8];
#pragma unroll
            for (int a = 0; a < 8; ++a) av[a] = As[kk][tr + 16 * a];
#pragma unroll
            for (int b = 0; b < 8; ++b) bv[b] = Bs[kk][tc + 16 * b];
#pragma unroll
            for (int a = 0; a < 8; ++a)
#pragma unroll
                for (int b = 0; b < 8; ++b) acc[a][b] += av[a] * bv[b];
        }
        __syncthreads();
    }
    // C's entries are loaded before any is stored, half of the tile at a time (a store may alias
    // a later load, so interleaved read-modify-writes would take one memory round trip each)
    const __amdgpu_buffer_rsrc_t rc = buf_rsrc(F.F + (r0 + bi) + (size_t)(r0 + bj) * lda);  // tile origin
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        double cv[4][8];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const int rl = bi + tr + 16 * (4 * h + a), cl = bj + tc + 16 * b;
                const bool ok = rl < nr && cl < nc && rl >= cl;
                const unsigned off = (unsigned)((rl - bi) + (size_t)(cl - bj) * lda) * 8u;
                cv[a][b] = buf_load_f64(rc, ok ? off : BUF_OOB);
            }
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const int rl = bi + tr + 16 * (4 * h + a), cl = bj + tc + 16 * b;
                if (rl < nr && cl < nc && rl >= cl)
                    A[(r0 + rl) + (size_t)(r0 + cl) * lda] = cv[a][b] - acc[4 * h + a][b];
            }
    }
}

// Deferred outer-block update in the reference's order.  update_trailing (factor.rs:1418-1526)
// subtracts each inner block's rank-nelim product from every fully-summed column beyond it; the
// columns beyond the current outer block are not read until their own outer block, so their
// updates are applied here, once per outer block, and still one inner block at a time: each
// entry of rows [obe, m) x columns [obe, p) becomes C - s_0 - s_1 - ..., s_b summed over block
// b's columns in ascending order from zero (gemm_sub_wlt), each subtraction rounded.  64 x 64
// tile per workgroup, each thread 4 x 4 entries kept in registers across the blocks.
__global__ __launch_bounds__(256, 3) void k_outer_exact(const FrontDev *__restrict__ fr,
                                                     const AptpState *__restrict__ st,
                                                     const TileItem *__restrict__ tiles,
                                                     double *const *__restrict__ wpp, unsigned ntiles) {
    const unsigned ti_ = tile_index(blockIdx.x, gridDim.x, true);
    if (ti_ >= ntiles) return;
    const TileItem t = tiles[ti_];
    const FrontDev &F = fr[t.front];
    const AptpState &S = st[t.aux];
    const int r0 = S.ob_start + S.ob_cols, nr = F.m - r0, nc = F.k - r0;
    const int nib = min(S.nib, MAX_OB_IB);
    if (nr <= 0 || nc <= 0 || S.kpos == S.ob_start) return;
    const int bi = t.ti * 64, bj = t.tj * 64;
    if (bi >= nr || bj >= nc || bi + 63 < bj) return;
    const size_t lda = F.m;
    const gdouble *A = gbl(F.F);
    // W = L D of the outer block's eliminated columns, rows [r0, m), leading dimension nr
    const gdouble *W = gbl(wpp[t.aux]);
    __shared__ double Ws[MAX_IB][65];
    __shared__ double Ls[MAX_IB][65];
    const int tid = threadIdx.x;
    const int tr = tid & 15, tc = tid >> 4;  // rows tr + 16a, columns tc + 16b
    const int lr = tid & 63, lk = tid >> 6;  // staging: row lr, columns lk + 4u
    // operands of one inner block prefetched into registers while the previous one computes
    double pw[MAX_IB / 4], pl[MAX_IB / 4];
    // range-checked buffer loads based at the block's first column (zero outside the tile): no
    // branch or select per load, so the prefetch stays in flight while the current block computes
    const int obs = S.ob_start;
    const bool wrow = bi + lr < nr, lrow = bj + lr < nc;
    auto prefetch = [&](int blk, int col0) {
        const int ne = S.ib_ne[blk];
        const __amdgpu_buffer_rsrc_t rw = buf_rsrc(wpp[t.aux] + bi + (size_t)(col0 - obs) * nr);
        const __amdgpu_buffer_rsrc_t rl = buf_rsrc(F.F + (r0 + bj) + (size_t)col0 * lda);
#pragma unroll
        for (int u = 0; u < MAX_IB / 4; ++u) {
            const int cc = lk + 4 * u;
            pw[u] = buf_load_f64(rw, (wrow && cc < ne) ? (unsigned)(lr + cc * nr) * 8u : BUF_OOB);
            pl[u] = buf_load_f64(rl, (lrow && cc < ne) ? (unsigned)(lr + cc * (int)lda) * 8u : BUF_OOB);
        }
    };
    int blk = 0, col0 = S.ob_start;
    while (blk < nib && S.ib_ne[blk] == 0) ++blk;
    if (blk < nib) prefetch(blk, col0);
    double c[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int rl = bi + tr + 16 * a, cl = bj + tc + 16 * b;
            c[a][b] = (rl < nr && cl < nc && rl >= cl) ? A[(r0 + rl) + (size_t)(r0 + cl) * lda] : 0.0;
        }
    while (blk < nib) {
        const int ne = S.ib_ne[blk];
        lds_barrier();  // the previous block's operands are consumed
#pragma unroll
        for (int u = 0; u < MAX_IB / 4; ++u) {
            const int cc = lk + 4 * u;
            if (cc < ne) {
                Ws[cc][lr] = pw[u];
                Ls[cc][lr] = pl[u];
            }
        }
        lds_barrier();
        int nblk = blk + 1;
        const int ncol0 = col0 + ne;
        while (nblk < nib && S.ib_ne[nblk] == 0) ++nblk;
        if (nblk < nib) prefetch(nblk, ncol0);
        double s[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) s[a][b] = 0.0;
        // two operand sets in turn: the next step's operands are read from LDS before the
        // current step's products, so their latency is covered (a row past ne, or row 0 after
        // the last, is read and unused)
        double w0[4], l0[4], w1[4], l1[4];
        auto rd = [&](double *w, double *l, int row) {
#pragma unroll
            for (int a = 0; a < 4; ++a) w[a] = Ws[row][tr + 16 * a];
#pragma unroll
            for (int b = 0; b < 4; ++b) l[b] = Ls[row][tc + 16 * b];
        };
        auto acc = [&](const double *w, const double *l) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) s[a][b] += w[a] * l[b];
        };
        rd(w0, l0, 0);
        int cc = 0;
#pragma unroll 1
        for (; cc + 1 < ne; cc += 2) {
            // scheduling barriers keep each read ahead of the products it overlaps
            rd(w1, l1, cc + 1);
            __builtin_amdgcn_sched_barrier(0);
            acc(w0, l0);
            __builtin_amdgcn_sched_barrier(0);
            rd(w0, l0, (cc + 2) & (MAX_IB - 1));
            __builtin_amdgcn_sched_barrier(0);
            acc(w1, l1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (cc < ne) acc(w0, l0);
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) c[a][b] -= s[a][b];
        blk = nblk;
        col0 = ncol0;
    }
    gdouble *Aw = gbl(F.F);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int rl = bi + tr + 16 * a, cl = bj + tc + 16 * b;
            if (rl < nr && cl < nc && rl >= cl) Aw[(r0 + rl) + (size_t)(r0 + cl) * lda] = c[a][b];
        }
}

constexpr int KF_CHUNK = 8192;  // doubles per k_keep_factor item

// Eliminated columns of a front held in the pool into its kept storage (the same column-major
// layout, lda = m): the first ne * m entries of the front.  One item = KF_CHUNK entries, 32 per
// thread, every load issued before the stores.
__global__ __launch_bounds__(256) void k_keep_factor(const FrontDev *__restrict__ fr,
                                                     const int2 *__restrict__ items) {
    const int2 it = items[blockIdx.x];
    const FrontDev &F = fr[it.x];
    const size_t n = (size_t)F.ne * F.m;
    const size_t base = (size_t)it.y * KF_CHUNK + threadIdx.x;
    if ((size_t)it.y * KF_CHUNK >= n) return;
    const gdouble *src = gbl((const double *)F.F);
    gdouble *dst = gbl(F.Lf);
    constexpr int U = KF_CHUNK / 256;
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const size_t i = base + (size_t)u * 256;
        v[u] = i < n ? src[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const size_t i = base + (size_t)u * 256;
        if (i < n) dst[i] = v[u];
    }
}

constexpr int RES_INTS = 10;  // per-front results of k_collect

// Per-front results (one workgroup of 256 threads per front): counts, inertia, max|L|, update
// flops, the solve's index map and the delayed columns.  Each loop issues the loads of COLB
// entries per thread before using any of them.
constexpr int COLB = 4;

__global__ __launch_bounds__(256) void k_collect(FrontDev *__restrict__ fr,
                                                 const int *__restrict__ flist,
                                                 const long long *__restrict__ doffs,
                                                 int *__restrict__ res, int *__restrict__ delayed) {
    const int li = blockIdx.x;
    const int f = flist[li];
    FrontDev &F = fr[f];
    const int ne = F.ne, k = F.k, m = F.m;
    const int tid = threadIdx.x;
    const gi8 *dkind = gbl(F.dkind);
    const gdouble *ddiag = gbl(F.ddiag), *doff = gbl(F.doff);
    // zero 1x1 pivots and the inertia of D (MixedDiagonal::compute_inertia, diagonal.rs:379-416)
    int z = 0, pos = 0, neg = 0, zer = 0;
    for (int c0 = tid; c0 < ne; c0 += 256 * COLB) {
        int kd[COLB];
        double a[COLB], b[COLB], cn[COLB];
#pragma unroll
        for (int u = 0; u < COLB; ++u) {
            const int c = c0 + 256 * u;
            kd[u] = (c < ne) ? dkind[c] : 0;
            a[u] = (c < ne) ? ddiag[c] : 0.0;
            b[u] = (c < ne) ? doff[c] : 0.0;
            cn[u] = (c + 1 < ne) ? ddiag[c + 1] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < COLB; ++u) {
            if (kd[u] == 1) {
                const double d = a[u];
                if (d > 0.0) ++pos;
                else if (d < 0.0) ++neg;
                else { ++zer; ++z; }
            } else if (kd[u] == 2) {
                const double det = a[u] * cn[u] - b[u] * b[u], tr = a[u] + cn[u];
                if (det > 0.0) {
                    if (tr > 0.0) pos += 2; else neg += 2;
                } else if (det < 0.0) {
                    ++pos; ++neg;
                } else if (tr > 0.0) {
                    ++pos; ++zer;
                } else if (tr < 0.0) {
                    ++neg; ++zer;
                } else {
                    zer += 2;
                }
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        z += __shfl_xor(z, o);
        pos += __shfl_xor(pos, o);
        neg += __shfl_xor(neg, o);
        zer += __shfl_xor(zer, o);
    }
    __shared__ int part[4][4];
    if ((tid & 63) == 0) {
        part[tid >> 6][0] = z;
        part[tid >> 6][1] = pos;
        part[tid >> 6][2] = neg;
        part[tid >> 6][3] = zer;
    }
    __syncthreads();
    if (tid == 0) {
        int *r = res + li * RES_INTS;
        r[0] = ne;
        r[1] = F.n1;
        r[2] = F.n2;
        r[7] = ((F.flags & FRONT_CHAIN_ERR) ? 1 : 0) | ((F.flags & FRONT_LA_ERR) ? 2 : 0);
        r[8] = (int)(unsigned)(F.obfail & 0xffffffffu);
        r[9] = (int)(unsigned)(F.obfail >> 32);
#pragma unroll
        for (int q = 0; q < 4; ++q) r[3 + q] = part[0][q] + part[1][q] + part[2][q] + part[3][q];
        unsigned long long *ml = (unsigned long long *)(res + RES_INTS * gridDim.x);
        ml[li] = F.max_l_bits;
        ((double *)(ml + gridDim.x))[li] = F.uflops;
    }
    int *dl = delayed + doffs[li];
    const gint *rows = gbl(F.rows), *perm = gbl(F.perm);
    gint *sidx = gbl(F.sidx);
    for (int i0 = tid; i0 < m; i0 += 256 * COLB) {
        int src[COLB], g[COLB];
#pragma unroll
        for (int u = 0; u < COLB; ++u) {
            const int i = i0 + 256 * u;
            src[u] = (i < k) ? perm[i] : i;
        }
#pragma unroll
        for (int u = 0; u < COLB; ++u) g[u] = (i0 + 256 * u < m) ? rows[src[u]] : 0;
#pragma unroll
        for (int u = 0; u < COLB; ++u) {
            const int i = i0 + 256 * u;
            if (i < m) {
                sidx[i] = g[u];
                if (i >= ne && i < k) dl[i - ne] = g[u];
            }
        }
    }
}

// ===========================================================================
// Host side
// ===========================================================================
namespace {

template <class T>
size_t stage_push(std::vector<char> &st, const T *data, size_t count) {
    size_t off = (st.size() + 255) / 256 * 256;
    st.resize(off + count * sizeof(T));
    if (count) std::memcpy(st.data() + off, data, count * sizeof(T));
    return off;
}

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

}  // namespace

void Prepared::build(const Symbolic &sym, const i64 *col_ptr, const i64 *row_idx, int nemin,
                     int small_leaf_threshold) {
    n = sym.n;
    nnz = col_ptr[n];
    perm_fwd = sym.perm_fwd;
    perm_inv = sym.perm_inv;
    sn_before = (long long)sym.sn.size();
    sns = amalgamate(sym.sn, nemin);
    merges = sn_before - (long long)sns.size();
    children = children_map(sns);
    int nodes = 0;
    small_leaf_subtrees = classify_small_leaf(sns, children, small_leaf_threshold, &nodes);
    small_leaf_nodes = nodes;
    const int ns = (int)sns.size();
    // height levels: a front's children are all in lower levels
    level_of.assign(ns, 0);
    int maxlv = 0;
    for (int s = 0; s < ns; ++s) {
        int lv = 0;
        for (int c : children[s]) lv = std::max(lv, level_of[c] + 1);
        level_of[s] = lv;
        maxlv = std::max(maxlv, lv);
    }
    levels.assign(ns ? maxlv + 1 : 0, {});
    for (int s = 0; s < ns; ++s) levels[level_of[s]].push_back(s);
    // amap (build_assembly_maps, numeric.rs:264-351), positions assuming no delays
    std::vector<int> g2l(n, -1);
    amap.clear();
    amap_off.assign(ns + 1, 0);
    for (int s = 0; s < ns; ++s) {
        const Supernode &S = sns[s];
        std::vector<int> rows;
        for (const ColRange &r : S.owned)
            for (int j = r.lo; j < r.hi; ++j) rows.push_back(j);
        const int total_owned = (int)rows.size();
        rows.insert(rows.end(), S.pattern.begin(), S.pattern.end());
        for (size_t i = 0; i < rows.size(); ++i) g2l[rows[i]] = (int)i;
        for (const ColRange &r : S.owned)
            for (int pj = r.lo; pj < r.hi; ++pj) {
                const int oc = perm_fwd[pj];
                const int lc = g2l[pj];
                for (i64 idx = col_ptr[oc]; idx < col_ptr[oc + 1]; ++idx) {
                    const int orow = (int)row_idx[idx];
                    if (orow < oc) {
                        const int peer = g2l[perm_inv[orow]];
                        if (peer >= 0 && peer < total_owned) continue;
                    }
                    const int gr = perm_inv[orow];
                    const int lr = g2l[gr];
                    if (lr < 0) continue;
                    AmapEntry e;
                    e.src = (unsigned)idx;
                    e.row = (unsigned)std::max(lr, lc);
                    e.col = (unsigned)std::min(lr, lc);
                    e.sr = (unsigned)gr;
                    e.sc = (unsigned)pj;
                    amap.push_back(e);
                }
            }
        for (int g : rows) g2l[g] = -1;
        amap_off[s + 1] = (i64)amap.size();
    }
    if (d_amap) { (void)hipFree(d_amap); d_amap = nullptr; }
    if (d_perm_fwd) { (void)hipFree(d_perm_fwd); d_perm_fwd = nullptr; }
    RV_HIP(hipMalloc(&d_amap, std::max<size_t>(1, amap.size()) * sizeof(AmapEntry)));
    if (!amap.empty())
        RV_HIP(hipMemcpy(d_amap, amap.data(), amap.size() * sizeof(AmapEntry), hipMemcpyHostToDevice));
    RV_HIP(hipMalloc(&d_perm_fwd, std::max<i64>(1, n) * sizeof(int)));
    if (n) RV_HIP(hipMemcpy(d_perm_fwd, perm_fwd.data(), n * sizeof(int), hipMemcpyHostToDevice));
}

Prepared::~Prepared() {
    if (d_amap) (void)hipFree(d_amap);
    if (d_perm_fwd) (void)hipFree(d_perm_fwd);
}

NumericGPU::NumericGPU(const Prepared *prep, const FactorOptions &opts, hipStream_t stream)
    : prep_(prep), o_(opts), stream_(stream) {
    const int ns = (int)prep->sns.size();
    RV_HIP(hipMalloc(&d_fr_, std::max(1, ns) * sizeof(FrontDev)));
    h_fr_.assign(ns, FrontDev());
    fprec_.assign(ns, (signed char)o_.update_precision);
    const char *ch = std::getenv("RV_APTP_CHAIN");
    chain_on_ = !(ch && std::strcmp(ch, "0") == 0);
    const char *la = std::getenv("RV_OUTER_LOOKAHEAD");
    la_on_ = !(la && std::strcmp(la, "0") == 0);
    const char *t64 = std::getenv("RV_OUTER_TILE64");
    outer_t64_ = !(t64 && std::strcmp(t64, "0") == 0);
    const char *kf = std::getenv("RV_KEEP_FRONTS");
    keep_fronts_ = kf && std::strcmp(kf, "1") == 0;
    obfail_.assign(ns, 0);
    pool_block_.assign(ns, -1);
}

size_t NumericGPU::chain_capacity(int ch) {
    int &cap = chain_cap_[ch == 64 ? 0 : 1];
    if (cap < 0) {
        int dev = 0, cus = 0, per = 0;
        RV_HIP(hipGetDevice(&dev));
        RV_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        if (ch == 64)
            RV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_aptp_outer<64>, 256, 0));
        else
            RV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_aptp_outer<128>, 256, 0));
        cap = per * cus;
    }
    return (size_t)cap;
}

void NumericGPU::set_front_precision(const signed char *prec) {
    std::vector<signed char> next(fprec_.size(), (signed char)o_.update_precision);
    if (prec) next.assign(prec, prec + fprec_.size());
    if (next != fprec_) {
        fprec_ = std::move(next);
        ++prec_gen_;  // every level plan is rebuilt at the next factorization
    }
}

void NumericGPU::drop_graph() {
    if (gexec_) (void)hipGraphExecDestroy(gexec_);
    if (graph_) (void)hipGraphDestroy(graph_);
    gexec_ = nullptr;
    graph_ = nullptr;
}

NumericGPU::~NumericGPU() {
    drop_graph();
    if (ev_fork_) (void)hipEventDestroy(ev_fork_);
    if (ev_join_) (void)hipEventDestroy(ev_join_);
    if (stream2_) (void)hipStreamDestroy(stream2_);
    if (d_fr_) (void)hipFree(d_fr_);
    for (auto &b : pin_blocks_) (void)hipHostFree(b.first);
    for (LevelPlan &L : plans_)
        for (auto &e : L.sev) {
            (void)hipEventDestroy(e.first);
            (void)hipEventDestroy(e.second);
        }
    if (d_sol_meta_) (void)hipFree(d_sol_meta_);
}

char *NumericGPU::pin_take(size_t bytes) {
    bytes = (bytes + 255) / 256 * 256;
    if (bytes == 0) bytes = 256;
    if (pin_cur_ < pin_blocks_.size() && pin_used_ + bytes <= pin_blocks_[pin_cur_].second) {
        char *p = pin_blocks_[pin_cur_].first + pin_used_;
        pin_used_ += bytes;
        return p;
    }
    if (pin_cur_ + 1 < pin_blocks_.size() && bytes <= pin_blocks_[pin_cur_ + 1].second) {
        ++pin_cur_;
        pin_used_ = bytes;
        return pin_blocks_[pin_cur_].first;
    }
    // a new block; blocks in use by transfers in flight are never freed here
    size_t total = 0;
    for (auto &b : pin_blocks_) total += b.second;
    const size_t sz = std::max({bytes, (size_t)4 << 20, total});
    char *p = nullptr;
    RV_HIP(hipHostMalloc((void **)&p, sz, hipHostMallocDefault));
    pin_blocks_.emplace_back(p, sz);
    pin_cur_ = pin_blocks_.size() - 1;
    pin_used_ = bytes;
    return p;
}

// Start of a factorization (no transfers in flight): merge the blocks into one.
void NumericGPU::pin_reset() {
    if (pin_blocks_.size() > 1) {
        size_t total = 0;
        for (auto &b : pin_blocks_) {
            total += b.second;
            (void)hipHostFree(b.first);
        }
        pin_blocks_.clear();
        char *p = nullptr;
        RV_HIP(hipHostMalloc((void **)&p, total, hipHostMallocDefault));
        pin_blocks_.emplace_back(p, total);
    }
    pin_cur_ = 0;
    pin_used_ = 0;
}

// Levels are planned and enqueued back to back with one synchronization at the end; each plan
// assumes the children's results the previous factorization produced (none delayed on the
// first).  Levels above the first one whose results differ from that assumption are planned
// again from the actual results and run one at a time.
void NumericGPU::factor(const double *d_val, const double *d_scaling) {
    const Prepared &P = *prep_;
    const int ns = (int)P.sns.size();
    const int nl = (int)P.levels.size();
    RV_HIP(hipStreamSynchronize(stream_));  // nothing of an earlier call may still be in flight
    if ((int)plans_.size() != nl) plans_.assign(nl, LevelPlan());
    for (const LevelPlan &L : plans_) belief_valid_ = belief_valid_ && L.valid;
    if (!belief_valid_) {
        for (LevelPlan &L : plans_) L.valid = false;
        ne_.assign(ns, 0);
        delayed_.assign(ns, {});
        m_.assign(ns, 0);
        k_.assign(ns, 0);
        rows_.assign(ns, {});
    }
    // the solve metadata depends only on each front's order, eliminated count and delayed
    // columns: keep it when a refactorization reproduces them
    const bool had_solve = solve_ready_ && belief_valid_;
    const bool had_solve_plans = belief_valid_;
    const std::vector<int> prev_ne = ne_, prev_m = m_;
    const std::vector<std::vector<int>> prev_delayed = delayed_;
    solve_ready_ = false;
    inv_valid_ = false;
    belief_valid_ = false;  // until this factorization completes
    n1_.assign(ns, 0); n2_.assign(ns, 0); zp_.assign(ns, 0);
    inert_.assign(ns, {0, 0, 0});
    maxl_.assign(ns, 0.0);
    times_ = PhaseTimes();
    pin_reset();
    // pass 1: every level enqueued on its plan
    std::vector<std::vector<int>> bel_ne(nl);
    std::vector<std::vector<std::vector<int>>> bel_del(nl);
    bool invalidate_rest = false;
    bool stable = graph_mode && had_solve_plans;
    for (int lv = 0; stable && lv < nl; ++lv)
        stable = plans_[lv].valid && plans_[lv].uploaded && plan_matches(lv);
    if (stable) {
        // every level runs on its existing plan: one launch of the captured level sequence
        // (captured on the first such call, and again whenever plans or inputs changed)
        if (!gexec_ || g_gen_ != plan_gen_ || g_val_ != d_val || g_scal_ != d_scaling) {
            drop_graph();
            const bool t = timing;
            timing = false;
            RV_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
            capturing_ = true;  // (one stream in the graph: no outer look-ahead)
            for (int lv = 0; lv < nl; ++lv) enqueue_level(lv, d_val, d_scaling);
            capturing_ = false;
            RV_HIP(hipStreamEndCapture(stream_, &graph_));
            timing = t;
            RV_HIP(hipGraphInstantiate(&gexec_, graph_, nullptr, nullptr, 0));
            g_gen_ = plan_gen_;
            g_val_ = d_val;
            g_scal_ = d_scaling;
        }
        for (int lv = 0; lv < nl; ++lv)
            for (int s : P.levels[lv]) {
                bel_ne[lv].push_back(ne_[s]);
                bel_del[lv].push_back(delayed_[s]);
            }
        RV_HIP(hipGraphLaunch(gexec_, stream_));
        ++graph_launches_;
    }
    for (int lv = 0; !stable && lv < nl; ++lv) {
        LevelPlan &L = plans_[lv];
        const bool rebuild = invalidate_rest || !L.valid || !plan_matches(lv);
        if (rebuild) {
            plan_level(lv, !invalidate_rest);
            invalidate_rest = true;  // the arena behind this level is handed out again
            // assume the rebuilt level delays nothing
            for (int s : P.levels[lv]) {
                ne_[s] = k_[s];
                delayed_[s].clear();
            }
        }
        for (int s : P.levels[lv]) {
            bel_ne[lv].push_back(ne_[s]);
            bel_del[lv].push_back(delayed_[s]);
        }
        enqueue_level(lv, d_val, d_scaling);
    }
    RV_HIP(hipStreamSynchronize(stream_));
    int first_bad = -1;
    for (int lv = 0; lv < nl && first_bad < 0; ++lv) {
        read_level(lv);
        const std::vector<int> &fr = P.levels[lv];
        for (size_t i = 0; i < fr.size(); ++i)
            if (ne_[fr[i]] != bel_ne[lv][i] || delayed_[fr[i]] != bel_del[lv][i]) first_bad = lv;
    }
    // pass 2 (only when a level's delays differed from the plans above it).  Pass 1's later
    // levels may have taken the pool blocks of contributions that the levels planned again read:
    // the levels up to first_bad run again first (same plans, same results).
    if (first_bad >= 0) {
        if (!keep_fronts_)
            for (int lv = 0; lv <= first_bad; ++lv) enqueue_level(lv, d_val, d_scaling);
        for (int lv = first_bad + 1; lv < nl; ++lv) {
            plan_level(lv, lv == first_bad + 1);
            enqueue_level(lv, d_val, d_scaling);
            RV_HIP(hipStreamSynchronize(stream_));
            read_level(lv);
        }
    }
    if (chain_err_) {
        // a wait of the persistent outer-block launch ran out (its workgroups were not all resident
        // at once): the results are void; factor again with the per-inner-block launches
        chain_err_ = false;
        la_err_ = false;
        chain_on_ = false;
        for (LevelPlan &L : plans_) L.valid = false;
        drop_graph();
        factor(d_val, d_scaling);
        return;
    }
    if (la_err_) {
        // an outer block planned without failed columns had some, and its trailing update ran
        // beside the delay swaps: the results are void; factor again in stream order (this
        // factorization's failures plan the next one)
        la_err_ = false;
        la_suspend_ = true;
        factor(d_val, d_scaling);
        la_suspend_ = false;
        return;
    }
    belief_valid_ = true;
    obfail_valid_ = true;
    // the solve plan holds the fronts' device addresses: any level planned since it was built
    // (plan_level hands out arena memory anew) makes it stale
    solve_ready_ = had_solve && prev_ne == ne_ && prev_m == m_ && prev_delayed == delayed_ &&
                   sol_plan_gen_ == plan_gen_;
    // the solve plan (and with it the workspace size rv_solve_scratch reports) follows every
    // factorization
    if (!solve_ready_) prepare_solve();
    // aggregate statistics (numeric.rs:929-1009)
    stats_ = FactorStats();
    stats_.sn_before = prep_->sn_before;
    stats_.sn_after = ns;
    stats_.merges = prep_->merges;
    stats_.small_leaf_subtrees = prep_->small_leaf_subtrees;
    stats_.small_leaf_nodes = prep_->small_leaf_nodes;
    for (int s = 0; s < ns; ++s) {
        stats_.total_1x1 += n1_[s];
        stats_.total_2x2 += n2_[s];
        stats_.total_delayed += k_[s] - ne_[s];
        stats_.max_front_size = std::max<long long>(stats_.max_front_size, m_[s]);
        if (prep_->sns[s].parent < 0 && ne_[s] < m_[s]) stats_.zero_pivots += k_[s] - ne_[s];
        stats_.zero_pivots += zp_[s];
    }
}

bool NumericGPU::plan_matches(int lv) const {
    const LevelPlan &L = plans_[lv];
    const Prepared &P = *prep_;
    if (L.prec_gen != prec_gen_) return false;
    size_t q = 0;
    for (int s : P.levels[lv])
        for (int c : P.children[s]) {
            if (q >= L.child_ne.size() || L.child_ne[q] != ne_[c] || L.child_del[q] != delayed_[c]) return false;
            ++q;
        }
    return q == L.child_ne.size();
}

// Pool blocks of level lv in placement order (largest first): every non-root front of at least
// 1 MiB is a block of its own, the smaller ones share one; each with the highest level of its
// fronts' parents (local indices into the level's front list, m per supernode).  None with
// keep_fronts_.
void NumericGPU::pool_groups(int lv, const std::vector<int> &m,
                             std::vector<std::pair<std::vector<int>, int>> *groups) const {
    const Prepared &P = *prep_;
    groups->clear();
    if (keep_fronts_) return;
    const std::vector<int> &fronts = P.levels[lv];
    std::vector<int> small;
    std::vector<std::pair<size_t, int>> big;
    int small_death = -1;
    size_t small_bytes = 0;
    for (int li = 0; li < (int)fronts.size(); ++li) {
        const int s = fronts[li];
        const int par = P.sns[s].parent;
        if (par < 0) continue;
        const size_t bytes = (size_t)m[s] * m[s] * sizeof(double);
        if (bytes >= ((size_t)1 << 20)) {
            big.emplace_back(bytes, li);
        } else {
            small.push_back(li);
            small_bytes += bytes;
            small_death = std::max(small_death, P.level_of[par]);
        }
    }
    std::stable_sort(big.begin(), big.end(), [](const std::pair<size_t, int> &a, const std::pair<size_t, int> &b) {
        return a.first > b.first;
    });
    bool small_done = small.empty();
    for (const auto &b : big) {
        if (!small_done && small_bytes >= b.first) {
            groups->emplace_back(small, small_death);
            small_done = true;
        }
        groups->emplace_back(std::vector<int>{b.second}, P.level_of[P.sns[fronts[b.second]].parent]);
    }
    if (!small_done) groups->emplace_back(small, small_death);
}

// Highest pool offset of a placement of every level's blocks at the fronts' sizes without
// delays: the size of the first pool chunk (plus a margin for fronts grown by delays).
size_t NumericGPU::pool_estimate() const {
    const Prepared &P = *prep_;
    const int ns = (int)P.sns.size();
    std::vector<int> m0(ns);
    for (int s = 0; s < ns; ++s) m0[s] = P.sns[s].n_owned() + (int)P.sns[s].pattern.size();
    FrontPool vp;
    vp.set_virtual();
    std::vector<std::pair<std::vector<int>, int>> groups;
    for (int lv = 0; lv < (int)P.levels.size(); ++lv) {
        pool_groups(lv, m0, &groups);
        for (const auto &g : groups) {
            size_t bytes = 0;
            for (int li : g.first) {
                const size_t mm = m0[P.levels[lv][li]];
                bytes += (mm * mm + 31) / 32 * 32 * sizeof(double);
            }
            vp.place(lv, g.second, bytes);
        }
    }
    return vp.top();
}

// reset_arena: the first level planned in a pass hands out the arena from its old mark (from
// the start for level 0); later levels of the pass allocate after it.
void NumericGPU::plan_level(int lv, bool reset_arena) {
    const Prepared &P = *prep_;
    LevelPlan &L = plans_[lv];
    if (reset_arena) {
        if (lv == 0) arena_.reset_keep();
        else arena_.reset_to(L.mark);
    }
    for (auto &e : L.sev) {
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    L = LevelPlan();
    L.mark = arena_.mark();
    ++plan_gen_;
    // working memory of a level's kernels (W panels, block backups, swap lines, APTP state) is
    // dead once the level's launches have run: every level takes it from the start of one
    // shared scratch arena, as the levels run in stream order
    scratch_.reset_keep();
    const std::vector<int> &fronts = P.levels[lv];
    const int nf = (int)fronts.size();
    const int nb = o_.outer_block_size, ib = o_.inner_block_size;
    L.prec_gen = prec_gen_;
    // updates beyond the current outer block: FP64 fronts defer them to k_outer_exact
    // (reference order, one pass per outer block; it holds at most MAX_OB_IB inner blocks, else
    // the inner blocks update every fully-summed column themselves); reduced-precision and
    // FP64-MFMA fronts (codes 1, 2, 4) to one rank-nb MFMA GEMM
    const bool exact_outer = cdiv(nb, ib) <= MAX_OB_IB;
    auto fp = [&](int s) { return (int)fprec_[s]; };
    auto deferred_f = [&](int s) { return fp(s) == 1 || fp(s) == 2 || fp(s) == 4; };
    for (int s : fronts)
        for (int c : P.children[s]) {
            L.child_ne.push_back(ne_[c]);
            L.child_del.push_back(delayed_[c]);
        }
    // ---- front structure (numeric.rs:1238-1262) ----
    size_t totF = 0, totM = 0, totK = 0;
    std::vector<int> ndel_in(nf);
    for (int li = 0; li < nf; ++li) {
        const int s = fronts[li];
        const Supernode &S = P.sns[s];
        std::vector<int> &rows = rows_[s];
        rows.clear();
        for (const ColRange &r : S.owned)
            for (int j = r.lo; j < r.hi; ++j) rows.push_back(j);
        const int nown = (int)rows.size();
        for (int c : P.children[s]) rows.insert(rows.end(), delayed_[c].begin(), delayed_[c].end());
        ndel_in[li] = (int)rows.size() - nown;
        const int k = (int)rows.size();
        rows.insert(rows.end(), S.pattern.begin(), S.pattern.end());
        m_[s] = (int)rows.size();
        k_[s] = k;
        totM += m_[s];
        totK += std::max(k, 1);
    }
    // ---- working fronts: roots (every front with keep_fronts_) in arena_, each with its factor
    // in place; the others in pool_ blocks that later levels take again once the parent level has
    // assembled them, their eliminated columns copied at the level's end to kept storage in arena_
    // (offsets in doubles rounded to 32: 256-byte aligned fronts) ----
    auto r32 = [](size_t x) { return (x + 31) / 32 * 32; };
    std::vector<double *> fptr(nf, nullptr), lptr(nf, nullptr);
    {
        pool_.drop_from(lv);
        if (!keep_fronts_ && pool_.bytes_reserved() == 0) {
            const size_t est = pool_estimate();
            pool_.reserve(est + est / 8);
        }
        std::vector<std::pair<std::vector<int>, int>> groups;
        pool_groups(lv, m_, &groups);
        for (int li = 0; li < nf; ++li) pool_block_[fronts[li]] = -1;
        for (const auto &g : groups) {
            size_t bytes = 0;
            for (int li : g.first) bytes += r32((size_t)m_[fronts[li]] * m_[fronts[li]]) * sizeof(double);
            const int id = pool_.place(lv, g.second, bytes);
            double *base = (double *)pool_.ptr(id);
            size_t o = 0;
            for (int li : g.first) {
                const int s = fronts[li];
                fptr[li] = base + o;
                o += r32((size_t)m_[s] * m_[s]);
                pool_block_[s] = id;
            }
        }
        size_t totF = 0, totL = 0;
        for (int li = 0; li < nf; ++li) {
            const int s = fronts[li];
            if (fptr[li]) totL += r32((size_t)m_[s] * k_[s]);
            else totF += r32((size_t)m_[s] * m_[s]);
        }
        double *Fbase = (double *)arena_.alloc(std::max<size_t>(totF + totL, 1) * sizeof(double));
        size_t fo = 0, lo = totF;
        for (int li = 0; li < nf; ++li) {
            const int s = fronts[li];
            if (fptr[li]) {
                lptr[li] = Fbase + lo;
                lo += r32((size_t)m_[s] * k_[s]);
            } else {
                fptr[li] = lptr[li] = Fbase + fo;
                fo += r32((size_t)m_[s] * m_[s]);
            }
        }
        L.Fbase = Fbase;
        L.totF = totF + totL;
    }
    // ---- device memory of the level ----
    int *ibase = (int *)arena_.alloc(std::max<size_t>(3 * totM, 1) * sizeof(int));
    int8_t *kbase = (int8_t *)arena_.alloc(std::max<size_t>(totK, 1));
    double *dbase = (double *)arena_.alloc(std::max<size_t>(2 * totK, 1) * sizeof(double));
    L.ibase = ibase;
    L.totM = totM;
    std::vector<FrontDev> lfr(nf);
    {
        size_t mo = 0, ko = 0;
        for (int li = 0; li < nf; ++li) {
            const int s = fronts[li];
            FrontDev d;
            std::memset(&d, 0, sizeof(d));
            d.F = fptr[li];
            d.Lf = lptr[li];
            d.rows = ibase + mo;
            d.perm = ibase + totM + mo;
            d.sidx = ibase + 2 * totM + mo;
            d.dkind = kbase + ko;
            d.ddiag = dbase + ko;
            d.doff = dbase + totK + ko;
            d.m = m_[s];
            d.k = k_[s];
            d.n_owned = P.sns[s].n_owned();
            d.ndelay_in = ndel_in[li];
            d.ne = 0;
            const bool tpp_whole = P.sns[s].in_small_leaf || d.k < ib;
            d.flags = (tpp_whole ? FRONT_TPP : 0) | (!deferred_f(s) && !exact_outer ? FRONT_ALLFS : 0) |
                      (fp(s) == 1 ? FRONT_W32 : 0);
            mo += d.m;
            ko += std::max(d.k, 1);
            lfr[li] = d;
            h_fr_[s] = d;
        }
    }
    // ---- work lists ----
    std::vector<ScatterChunk> sch;
    std::vector<int> tpp_list, aptp_list;
    for (int li = 0; li < nf; ++li) {
        const int s = fronts[li];
        for (i64 b = P.amap_off[s]; b < P.amap_off[s + 1]; b += 256)
            sch.push_back(ScatterChunk{s, (int)b, (int)std::min<i64>(b + 256, P.amap_off[s + 1]), 0});
        if (lfr[li].flags & FRONT_TPP) tpp_list.push_back(s);
        else aptp_list.push_back(s);
    }
    // extend-add maps: contribution rows of each child -> parent local rows.  Children whose rows
    // have none in common touch no common entry of the parent and share a launch; the rest keep
    // their order: a child's round follows the last round of any row of its own, so every entry
    // sums its children in reference order.  (KKT side 64: 316 launches with one per child
    // ordinal, 83 so, about 5 us each; step 8.6 -> 6.9 ms.)
    int nrounds = 0;
    std::vector<unsigned> maps;
    struct EaPending { int child, parent, round, size, cne; size_t mapoff; int skip; };
    std::vector<EaPending> eap;
    {
        std::vector<int> g2l;
        g2l.assign(P.n, -1);
        for (int li = 0; li < nf; ++li) {
            const int s = fronts[li];
            const std::vector<int> &prow = rows_[s];
            for (size_t i = 0; i < prow.size(); ++i) g2l[prow[i]] = (int)i;
            std::vector<int> next_round(prow.size(), 0);
            const std::vector<int> &ch = P.children[s];
            for (size_t ci = 0; ci < ch.size(); ++ci) {
                const int c = ch[ci];
                const int sz = m_[c] - ne_[c];
                if (sz == 0) continue;  // fully eliminated child: no contribution
                EaPending e;
                e.child = c; e.parent = s; e.round = 0; e.size = sz; e.cne = ne_[c];
                e.mapoff = maps.size();
                for (int g : delayed_[c]) maps.push_back((unsigned)g2l[g]);
                for (int g : P.sns[c].pattern) maps.push_back((unsigned)g2l[g]);
                for (size_t q = e.mapoff; q < maps.size(); ++q)
                    if ((int)maps[q] < 0 || (int)maps[q] >= (int)prow.size())
                        throw std::runtime_error("contribution row of supernode " + std::to_string(c) +
                                                 " is not in its parent's front");
                for (size_t q = e.mapoff; q < maps.size(); ++q) e.round = std::max(e.round, next_round[maps[q]]);
                for (size_t q = e.mapoff; q < maps.size(); ++q) next_round[maps[q]] = e.round + 1;
                nrounds = std::max(nrounds, e.round + 1);
                const bool g2l_path = !delayed_[c].empty() || ndel_in[li] > 0;
                e.skip = (P.sns[s].in_small_leaf || g2l_path) ? 1 : 0;
                eap.push_back(e);
            }
            for (int g : prow) g2l[g] = -1;
        }
    }
    // ---- staging blob ----
    std::vector<char> &stg = L.stage;
    std::vector<int> ids(fronts.begin(), fronts.end());
    L.nf = nf;
    L.o_ids = stage_push(stg, ids.data(), ids.size());
    L.o_lfr = stage_push(stg, lfr.data(), lfr.size());
    {
        std::vector<int2> zitems;
        for (int li = 0; li < nf; ++li)
            for (int c = 0; c < lfr[li].m; c += ZCOLS) zitems.push_back(make_int2(li, c));
        L.o_zl = stage_push(stg, zitems.data(), zitems.size());
        L.nzl = zitems.size();
        // eliminated columns of the pooled fronts into their kept storage (supernode, chunk)
        std::vector<int2> kitems;
        for (int li = 0; li < nf; ++li)
            if (lfr[li].Lf != lfr[li].F)
                for (size_t c = 0; c * KF_CHUNK < (size_t)lfr[li].m * lfr[li].k; ++c)
                    kitems.push_back(make_int2(fronts[li], (int)c));
        L.o_kf = stage_push(stg, kitems.data(), kitems.size());
        L.nkf = kitems.size();
    }
    std::vector<int> rowsflat;
    rowsflat.reserve(totM);
    for (int s : fronts) rowsflat.insert(rowsflat.end(), rows_[s].begin(), rows_[s].end());
    L.o_rows = stage_push(stg, rowsflat.data(), rowsflat.size());
    L.o_sch = stage_push(stg, sch.data(), sch.size());
    L.nsch = sch.size();
    const size_t o_maps = stage_push(stg, maps.data(), maps.size());
    auto tpp_need = [&](int s) { return tpp_lds_bytes(m_[s], k_[s]); };
    auto tpp_wave = [&](int s) { return m_[s] <= 64 && tpp_need(s) <= TPP_LDS_WAVE; };
    auto tpp_mid = [&](int s) { return tpp_need(s) > TPP_LDS_HALF && tpp_need(s) <= TPP_LDS_MAX; };
    const bool waves = std::count_if(tpp_list.begin(), tpp_list.end(), tpp_wave) > TPP_WAVE_MIN;
    const bool mids = std::count_if(tpp_list.begin(), tpp_list.end(), tpp_mid) > TPP_MID_MIN;
    auto tpp_class = [&](int s) {
        return waves && tpp_wave(s) ? TPP_WAVE : tpp_need(s) <= TPP_LDS_SMALL ? TPP_SMALL : mids && tpp_mid(s) ? TPP_MID : TPP_WIDE;
    };
    std::stable_sort(tpp_list.begin(), tpp_list.end(), [&](int a, int b) { return tpp_class(a) < tpp_class(b); });
    std::fill(L.ntpp, L.ntpp + 4, 0);
    std::fill(L.tpp_lds, L.tpp_lds + 4, 0);
    for (int s : tpp_list) {
        const int c = tpp_class(s);
        ++L.ntpp[c];
        if (tpp_need(s) <= TPP_LDS_MAX) L.tpp_lds[c] = std::max(L.tpp_lds[c], tpp_need(s));
    }
    L.tpp_lds[TPP_MID] = std::min(L.tpp_lds[TPP_MID], TPP_LDS_SMALL);
    L.o_tpp = stage_push(stg, tpp_list.data(), tpp_list.size());
    L.o_aptp = stage_push(stg, aptp_list.data(), aptp_list.size());
    // extend-add items per round; map fields hold blob offsets until the device copy exists
    std::vector<std::vector<EaItem>> ea_rounds(nrounds);
    for (const EaPending &e : eap) {
        const int nt = cdiv(e.size, 64);
        for (int ti = 0; ti < nt; ++ti)
            for (int tj = 0; tj <= ti; ++tj) {
                EaItem it;
                it.child = e.child; it.parent = e.parent; it.ti = ti; it.tj = tj;
                it.map = (const unsigned *)(uintptr_t)(o_maps + e.mapoff * sizeof(unsigned));
                it.skip_zero = e.skip; it.cne = e.cne;
                ea_rounds[e.round].push_back(it);
            }
    }
    L.o_ea.resize(nrounds);
    L.n_ea.resize(nrounds);
    for (int r = 0; r < nrounds; ++r) {
        L.o_ea[r] = stage_push(stg, ea_rounds[r].data(), ea_rounds[r].size());
        L.n_ea[r] = ea_rounds[r].size();
    }
    // APTP item lists
    const int na = (int)aptp_list.size();
    L.na = na;
    // work items carry the front's index next to its APTP slot: the kernels read the front
    // descriptor without a dependent load of the slot list
    std::vector<int4> k2items;
    std::vector<int4> k3items;
    // the look-ahead workgroups first, so they are dispatched with the first wave of workgroups
    for (int li = 0; li < na; ++li)
        if (k_[aptp_list[li]] > ib) k3items.push_back(make_int4(li, 0, LOOKAHEAD_Q, aptp_list[li]));
    int max_outer = 0;
    for (int li = 0; li < na; ++li) {
        const int s = aptp_list[li];
        const int m = m_[s], p = k_[s];
        for (int c = 0; c < cdiv(m, 256); ++c) k2items.push_back(make_int4(li, c, s, 0));
        const int qmax = 1 + cdiv((deferred_f(s) || exact_outer) ? std::min(p, nb) : p, 32);
        for (int rt = 0; rt < cdiv(m, 64); ++rt)
            for (int q = 0; q < qmax; ++q) k3items.push_back(make_int4(li, rt, q, s));
        const int nouter = p > nb ? cdiv(p, nb) : 1;
        max_outer = std::max(max_outer, nouter);
    }
    L.max_outer = max_outer;
    L.o_k2 = stage_push(stg, k2items.data(), k2items.size());
    L.nk2 = k2items.size();
    L.o_k3 = stage_push(stg, k3items.data(), k3items.size());
    L.nk3 = k3items.size();
    L.ninner.assign(max_outer, 0);
    for (int ob = 0; ob < max_outer; ++ob)
        for (int s : aptp_list) {
            const int p = k_[s];
            const bool two = p > nb;
            const int nouter = two ? cdiv(p, nb) : 1;
            if (ob >= nouter) continue;
            const int obcols = two ? std::min(nb, p - ob * nb) : p;
            L.ninner[ob] = std::max(L.ninner[ob], cdiv(obcols, ib));
        }
    // one persistent launch per outer block when every workgroup of the level's largest one
    // (outer block 0: leader + panels of CH rows per front) is resident at once and the inner
    // blocks fit the launch's records
    L.chain_ch = 0;
    L.o_chain.clear();
    L.n_chain.clear();
    L.dC = nullptr;
    // (at most CHAIN_MAX_IT inner blocks per outer block also means no front of the level updates every
    // fully-summed column from its inner blocks: exact_outer holds)
    if (na > 0 && chain_on_ && cdiv(nb, ib) <= CHAIN_MAX_IT && ib <= MAX_IB) {
        for (int ch : {64, 128}) {
            size_t tot = 0;
            for (int s : aptp_list) tot += 1 + cdiv(m_[s], ch);
            if (tot <= chain_capacity(ch)) {
                L.chain_ch = ch;
                break;
            }
        }
    }
    if (L.chain_ch) {
        const int ch = L.chain_ch;
        L.o_chain.assign(max_outer, 0);
        L.n_chain.assign(max_outer, 0);
        for (int ob = 0; ob < max_outer; ++ob) {
            // leaders first, then the panels front by front
            std::vector<int4> items;
            std::vector<int> npan(na, 0);
            for (int li = 0; li < na; ++li) {
                const int s = aptp_list[li], p = k_[s];
                const int nouter = p > nb ? cdiv(p, nb) : 1;
                if (ob >= nouter) continue;
                npan[li] = cdiv(m_[s] - ob * nb, ch);
                items.push_back(make_int4(li, 0, s, npan[li]));
            }
            for (int li = 0; li < na; ++li)
                for (int q = 0; q < npan[li]; ++q) items.push_back(make_int4(li, 1 + q, aptp_list[li], npan[li]));
            L.o_chain[ob] = stage_push(stg, items.data(), items.size());
            L.n_chain[ob] = items.size();
        }
        L.dC = (ChainSync *)scratch_.alloc((size_t)na * sizeof(ChainSync));
    }
    // contribution GEMM tiles (mode 0), one list per update precision
    std::array<std::vector<TileItem>, 4> ctiles;
    for (int li = 0; li < nf; ++li) {
        const int s = fronts[li];
        if (P.sns[s].parent < 0) continue;
        const int nfs = m_[s] - k_[s];
        if (nfs <= 0) continue;
        const int nt = cdiv(nfs, 128);
        for (int ti = 0; ti < nt; ++ti)
            for (int tj = 0; tj <= ti; ++tj) ctiles[fp(s) == 4 ? 0 : fp(s)].push_back(TileItem{s, ti, tj, li});
    }
    for (int q = 0; q < 4; ++q) {
        L.o_ct[q] = stage_push(stg, ctiles[q].data(), ctiles[q].size());
        L.nct[q] = ctiles[q].size();
    }
    // W = L D buffers and their k_form_ld items: mode 0 per level front, mode 1 per APTP front
    std::vector<double *> wp0(nf, nullptr), wp1(aptp_list.size(), nullptr), wp1b(aptp_list.size(), nullptr);
    std::vector<int4> f0items, f1items;
    for (int li = 0; li < nf; ++li) {
        const int s = fronts[li];
        if (P.sns[s].parent < 0) continue;
        const int nfs = m_[s] - k_[s];
        if (nfs <= 0 || k_[s] <= 0) continue;
        wp0[li] = (double *)scratch_.alloc((size_t)nfs * k_[s] * sizeof(double));
        for (int rc = 0; rc < cdiv(nfs, 256); ++rc)
            for (int cc = 0; cc < cdiv(k_[s], FC); ++cc) f0items.push_back(make_int4(s, li, rc, cc));
    }
    for (size_t li = 0; li < aptp_list.size(); ++li) {
        const int s = aptp_list[li];
        if (k_[s] <= nb || !(deferred_f(s) || exact_outer)) continue;
        wp1[li] = (double *)scratch_.alloc((size_t)m_[s] * nb * sizeof(double));
        wp1b[li] = (double *)scratch_.alloc((size_t)m_[s] * nb * sizeof(double));
        for (int rc = 0; rc < cdiv(m_[s], 256); ++rc)
            for (int cc = 0; cc < cdiv(nb, FC); ++cc) f1items.push_back(make_int4(s, (int)li, rc, cc));
    }
    L.o_wp0 = stage_push(stg, wp0.data(), wp0.size());
    L.o_wp1 = stage_push(stg, wp1.data(), wp1.size());
    L.o_wp1b = stage_push(stg, wp1b.data(), wp1b.size());
    L.o_f0 = stage_push(stg, f0items.data(), f0items.size());
    L.nf0 = f0items.size();
    L.o_f1 = stage_push(stg, f1items.data(), f1items.size());
    L.nf1 = f1items.size();
    L.ota64 = outer_t64_ && nb % 128 == 0;
    // outer-update tiles (mode 1) per outer block index and kind (exact, FP32, BF16, FP64 MFMA):
    // the tiles in the next outer block's columns first (otiles), then the rest (otiles_b)
    std::vector<std::array<std::vector<TileItem>, 4>> otiles(max_outer), otiles_b(max_outer);
    for (int li = 0; li < na; ++li) {
        const int s = aptp_list[li];
        const int m = m_[s], p = k_[s];
        const bool dfr = deferred_f(s);
        if (p <= nb || !(dfr || exact_outer)) continue;
        const int nouter = cdiv(p, nb);
        const int kind = dfr ? (fp(s) == 4 ? 3 : fp(s)) : 0;
        const int T = dfr ? 128 : 64;  // k_schur tiles / k_outer_exact tiles
        // the next block's columns in 64 x 64 k_schur tiles (FP32, FP64 MFMA; see L.ota64)
        const int TA = (dfr && L.ota64 && kind != 2) ? 64 : T;
        // every outer block: columns beyond it hold later blocks and earlier blocks' delays
        for (int ob = 0; ob < nouter; ++ob) {
            const int obcols = std::min(nb, p - ob * nb);
            const int nr = m - obcols, nc = p - obcols;
            if (nc <= 0) continue;
            const int ntr = cdiv(nr, T), ntc = cdiv(nc, T);
            if (TA != T) {
                // (nb a multiple of 128: both tilings split the columns at nb)
                for (int ti = 0; ti < cdiv(nr, TA); ++ti)
                    for (int tj = 0; tj <= std::min(ti, std::min(cdiv(nc, TA), nb / TA) - 1); ++tj)
                        otiles[ob][kind].push_back(TileItem{s, ti, tj, li});
                for (int ti = 0; ti < ntr; ++ti)
                    for (int tj = nb / T; tj <= std::min(ti, ntc - 1); ++tj)
                        otiles_b[ob][kind].push_back(TileItem{s, ti, tj, li});
                continue;
            }
            for (int ti = 0; ti < ntr; ++ti)
                for (int tj = 0; tj <= std::min(ti, ntc - 1); ++tj)
                    (tj < cdiv(nb, T) ? otiles : otiles_b)[ob][kind].push_back(TileItem{s, ti, tj, li});
        }
    }
    L.o_ot.resize(max_outer);
    L.n_ot.resize(max_outer);
    L.na_ot.resize(max_outer);
    for (int ob = 0; ob < max_outer; ++ob)
        for (int q = 0; q < 4; ++q) {
            L.na_ot[ob][q] = otiles[ob][q].size();
            otiles[ob][q].insert(otiles[ob][q].end(), otiles_b[ob][q].begin(), otiles_b[ob][q].end());
            L.o_ot[ob][q] = stage_push(stg, otiles[ob][q].data(), otiles[ob][q].size());
            L.n_ot[ob][q] = otiles[ob][q].size();
        }
    L.doffs.assign(nf + 1, 0);
    for (int li = 0; li < nf; ++li) L.doffs[li + 1] = L.doffs[li] + std::max(k_[fronts[li]], 1);
    L.o_doffs = stage_push(stg, L.doffs.data(), L.doffs.size());
    // APTP state and scratch: backup (m x ib), touched lines' crossings of a permutation
    if (na > 0) {
        std::vector<AptpState> hs(na);
        for (int li = 0; li < na; ++li) {
            AptpState &S = hs[li];
            std::memset(&S, 0, sizeof(S));
            S.fail_min = INT_MAX;
            const int m = m_[aptp_list[li]];
            S.backup = (double *)scratch_.alloc((size_t)m * ib * sizeof(double));
            S.blkcopy = (double *)scratch_.alloc((size_t)MAX_IB * MAX_IB * sizeof(double));
            S.swapbuf = (double *)scratch_.alloc((size_t)4 * MAX_IB * MAX_IB * sizeof(double));
        }
        L.dS = (AptpState *)scratch_.alloc((size_t)na * sizeof(AptpState));
        L.dSnap[0] = (AptpState *)scratch_.alloc((size_t)na * sizeof(AptpState));
        L.dSnap[1] = (AptpState *)scratch_.alloc((size_t)na * sizeof(AptpState));
        L.dleft = (int *)scratch_.alloc((size_t)(na + 1) * sizeof(int));
        L.o_hs = stage_push(stg, hs.data(), hs.size());
    }
    // device copy of the blob; extend-add map fields become device addresses
    L.dstage = (char *)arena_.alloc(stg.size());
    for (int r = 0; r < nrounds; ++r) {
        EaItem *items = (EaItem *)(stg.data() + L.o_ea[r]);
        for (size_t i = 0; i < L.n_ea[r]; ++i)
            items[i].map = (const unsigned *)(L.dstage + (size_t)(uintptr_t)items[i].map);
    }
    // k_collect results: ints, max|L| bits, update flops, then the delayed columns
    const size_t rbytes = (size_t)nf * RES_INTS * sizeof(int) + (size_t)nf * 16;
    L.res_del_off = (rbytes + 255) / 256 * 256;
    L.res_bytes = L.res_del_off + (size_t)L.doffs[nf] * sizeof(int);
    L.dres = (char *)arena_.alloc(L.res_bytes);
    L.valid = true;
}

void NumericGPU::ensure_stream2() {
    if (stream2_) return;
    RV_HIP(hipStreamCreate(&stream2_));
    RV_HIP(hipEventCreateWithFlags(&ev_fork_, hipEventDisableTiming));
    RV_HIP(hipEventCreateWithFlags(&ev_join_, hipEventDisableTiming));
}

void NumericGPU::enqueue_level(int lv, const double *d_val, const double *d_scaling) {
    const Prepared &P = *prep_;
    LevelPlan &L = plans_[lv];
    const int nb = o_.outer_block_size, ib = o_.inner_block_size;
    if (!L.uploaded) {
        char *hp = pin_take(L.stage.size());
        std::memcpy(hp, L.stage.data(), L.stage.size());
        RV_HIP(hipMemcpyAsync(L.dstage, hp, L.stage.size(), hipMemcpyHostToDevice, stream_));
        L.uploaded = true;
    }
    for (auto &e : L.sev) {
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    L.sev.clear();
    L.sev_contrib.clear();
    auto D = [&](size_t off) { return L.dstage + off; };
    // Schur GEMM launches, bracketed by HIP events on their stream when timing is on
    auto timed_schur = [&](hipStream_t sm, int prec, size_t ntiles, const TileItem *tl, AptpState *stp, int mode,
                           double *const *wpp, bool t64 = false) {
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (timing) {
            RV_HIP(hipEventCreate(&e0));
            RV_HIP(hipEventCreate(&e1));
            RV_HIP(hipEventRecord(e0, sm));
        }
        const dim3 grid(mode == 1 ? spread_grid(ntiles) : (unsigned)ntiles), block(256);
        const unsigned nt = (unsigned)ntiles;
        if (prec == 3)
            hipLaunchKernelGGL(k_schur_exact, grid, block, 0, sm, d_fr_, (const AptpState *)stp, tl, mode, wpp, nt);
        else if (prec == 1 && t64)
            hipLaunchKernelGGL((k_schur<1, 64>), grid, block, 0, sm, d_fr_, (const AptpState *)stp, tl, mode, wpp, nt);
        else if (prec == 1)
            hipLaunchKernelGGL(k_schur<1>, grid, block, 0, sm, d_fr_, (const AptpState *)stp, tl, mode, wpp, nt);
        else if (prec == 2)
            hipLaunchKernelGGL(k_schur<2>, grid, block, 0, sm, d_fr_, (const AptpState *)stp, tl, mode, wpp, nt);
        else if (t64)
            hipLaunchKernelGGL((k_schur<0, 64>), grid, block, 0, sm, d_fr_, (const AptpState *)stp, tl, mode, wpp, nt);
        else
            hipLaunchKernelGGL(k_schur<0>, grid, block, 0, sm, d_fr_, (const AptpState *)stp, tl, mode, wpp, nt);
        if (timing) {
            RV_HIP(hipEventRecord(e1, sm));
            L.sev.emplace_back(e0, e1);
            L.sev_contrib.push_back(mode == 0 ? 1 : 0);
        }
    };
    // deferred exact outer updates, timed with the Schur GEMMs
    auto timed_outer = [&](hipStream_t sm, size_t ntiles, const TileItem *tl, AptpState *stp, double *const *wpp) {
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (timing) {
            RV_HIP(hipEventCreate(&e0));
            RV_HIP(hipEventCreate(&e1));
            RV_HIP(hipEventRecord(e0, sm));
        }
        hipLaunchKernelGGL(k_outer_exact, dim3(spread_grid(ntiles)), dim3(256), 0, sm, d_fr_,
                           (const AptpState *)stp, tl, wpp, (unsigned)ntiles);
        if (timing) {
            RV_HIP(hipEventRecord(e1, sm));
            L.sev.emplace_back(e0, e1);
            L.sev_contrib.push_back(0);
        }
    };
    // outer look-ahead for this level: the trailing update of outer block ob may run on stream2_
    // beside block ob + 1 when no front of the level had failed columns in block ob in the last
    // factorization (failed columns are swapped into the trailing columns at the block's end)
    auto lookahead_ok = [&](int ob) {
        if (!la_on_ || la_suspend_ || capturing_ || !obfail_valid_ || ob + 1 >= L.max_outer) return false;
        const int *al = (const int *)(L.stage.data() + L.o_aptp);
        for (int li = 0; li < L.na; ++li)
            if (ob >= 63 || ((obfail_[al[li]] >> ob) & 1ull)) return false;
        return true;
    };
    const int nf = L.nf, na = L.na;
    // ---- lower triangles zeroed, per-front descriptors, perm, rows: one launch ----
    {
        const long long nrows = (long long)L.totM;
        const unsigned nb_setup = (unsigned)(L.nzl + cdiv(nf, 256) + nf + (nrows + ROWCOPY - 1) / ROWCOPY);
        hipLaunchKernelGGL(k_level_setup, dim3(nb_setup), dim3(256), 0, stream_, d_fr_, (const int *)D(L.o_ids),
                           (const FrontDev *)D(L.o_lfr), nf, (const int2 *)D(L.o_zl), (int)L.nzl, (int *)L.ibase,
                           (const int *)D(L.o_rows), nrows);
    }
    // ---- assembly ----
    if (L.nsch)
        hipLaunchKernelGGL(k_scatter_orig, dim3((unsigned)L.nsch), dim3(256), 0, stream_, d_fr_,
                           (const ScatterChunk *)D(L.o_sch), P.d_amap, d_val, d_scaling);
    for (size_t r = 0; r < L.n_ea.size(); ++r)
        if (L.n_ea[r])
            hipLaunchKernelGGL(k_extend_add, dim3((unsigned)L.n_ea[r]), dim3(256), 0, stream_, d_fr_,
                               (const EaItem *)D(L.o_ea[r]));
    // ---- TPP fronts ----
    // (launches of their own: one wide front does not take the other fronts' residency)
    const int *tpp = (const int *)D(L.o_tpp);
    for (int c = 0; c < 4; ++c) {
        const unsigned n = (unsigned)L.ntpp[c], lds = (unsigned)L.tpp_lds[c];
        if (!n) continue;
        const auto kernel = c == TPP_WAVE ? k_tpp<64, 2, false> : c == TPP_MID ? k_tpp<128, 4, true> : k_tpp<256, 4, false>;
        hipLaunchKernelGGL(kernel, dim3(n), dim3(c == TPP_WAVE ? 64 : c == TPP_MID ? 128 : 256), lds, stream_, d_fr_, tpp,
                           o_.threshold, o_.small, lds);
        tpp += n;
    }
    // ---- APTP fronts ----
    if (na > 0) {
        AptpState *dS = L.dS;
        const int *dl = (const int *)D(L.o_aptp);
        bool la_pending = false;  // a trailing update runs on stream2_ (joined before the next one)
        for (int ob = 0; ob < L.max_outer; ++ob) {
            if (ob == 0)
                hipLaunchKernelGGL(k_outer_first, dim3(na), dim3(256), 0, stream_, d_fr_, dS,
                                   (const AptpState *)D(L.o_hs), dl, nb, ib, L.dC, L.dleft);
            if (L.chain_ch && L.n_chain[ob]) ++chain_launches_;
            if (L.chain_ch == 64 && L.n_chain[ob])
                hipLaunchKernelGGL(k_aptp_outer<64>, dim3((unsigned)L.n_chain[ob]), dim3(256), 0, stream_, d_fr_,
                                   dS, L.dC, (const int4 *)D(L.o_chain[ob]), nb, ib, o_.small, o_.threshold);
            else if (L.chain_ch == 128 && L.n_chain[ob])
                hipLaunchKernelGGL(k_aptp_outer<128>, dim3((unsigned)L.n_chain[ob]), dim3(256), 0, stream_, d_fr_,
                                   dS, L.dC, (const int4 *)D(L.o_chain[ob]), nb, ib, o_.small, o_.threshold);
            for (int it = 0; !L.chain_ch && it < L.ninner[ob]; ++it) {
                hipLaunchKernelGGL(k_block_apply, dim3((unsigned)L.nk2), dim3(256), 0, stream_, d_fr_, dS,
                                   dl, (const int4 *)D(L.o_k2), ob, it, nb, ib, o_.small, o_.threshold);
                hipLaunchKernelGGL(k_block_update, dim3((unsigned)L.nk3), dim3(256), 0, stream_, d_fr_,
                                   dS, dl, (const int4 *)D(L.o_k3), ob, it, nb, ib, o_.small);
                hipLaunchKernelGGL(k_block_finish, dim3(na), dim3(256), 0, stream_, d_fr_, dS, dl, ob,
                                   it, nb, ib);
            }
            // W of block ob in one of two buffers by parity: the trailing update of block ob - 1
            // may still read the other
            const int par = ob & 1;
            double *const *wpp = (double *const *)D(par ? L.o_wp1b : L.o_wp1);
            size_t n_rest = 0;
            for (int q = 0; q < 4; ++q) n_rest += L.n_ot[ob][q] - L.na_ot[ob][q];
            const bool la = n_rest > 0 && lookahead_ok(ob);
            if (la) ensure_stream2();
            // W of block ob; with look-ahead also the states as block ob left them (k_outer_next
            // moves them on to block ob + 1 while the rest of this update still runs)
            if ((L.n_ot[ob][0] || L.n_ot[ob][1] || L.n_ot[ob][2] || L.n_ot[ob][3]) && L.nf1)
                hipLaunchKernelGGL(k_form_ld, dim3((unsigned)L.nf1), dim3(256), 0, stream_, d_fr_, dS,
                                   (const int4 *)D(L.o_f1), 1, wpp, la ? L.dSnap[par] : (AptpState *)nullptr);
            // the columns of block ob + 1 on from here received block ob - 1's trailing update
            if (la_pending) {
                RV_HIP(hipStreamWaitEvent(stream_, ev_join_, 0));
                la_pending = false;
            }
            // next block's columns (all columns without look-ahead) here, the rest beside block ob + 1
            // (kind 3: FP64 MFMA, k_schur<0>); with L.ota64 the next block's columns come in 64 x 64
            // tiles (FP32, FP64 MFMA) and the rest in 128 x 128 tiles, one launch each
            for (int q = 1; q <= 3; ++q) {
                const bool t64 = L.ota64 && q != 2;
                const size_t na_q = L.na_ot[ob][q], n_q = L.n_ot[ob][q];
                const size_t nhere = (la || t64) ? na_q : n_q;
                if (nhere) timed_schur(stream_, q == 3 ? 0 : q, nhere, (const TileItem *)D(L.o_ot[ob][q]), dS, 1, wpp, t64);
                if (!la && t64 && n_q > na_q)
                    timed_schur(stream_, q == 3 ? 0 : q, n_q - na_q, (const TileItem *)D(L.o_ot[ob][q]) + na_q, dS, 1, wpp);
            }
            {
                const size_t nhere = la ? L.na_ot[ob][0] : L.n_ot[ob][0];
                if (nhere) timed_outer(stream_, nhere, (const TileItem *)D(L.o_ot[ob][0]), dS, wpp);
            }
            if (ob + 1 < L.max_outer)
                hipLaunchKernelGGL(k_outer_next, dim3(na), dim3(512), 0, stream_, d_fr_, dS, dl, ob, nb, ib, L.dC,
                                   la ? 1 : 0, L.dleft);
            else
                hipLaunchKernelGGL(k_outer_end, dim3(na), dim3(256), 0, stream_, d_fr_, dS, dl, ob, nb, L.dleft);
            if (la) {
                // forked once block ob + 1 can start, so that its persistent launch and this update
                // begin dispatching together (an update dispatched first would hold every slot)
                RV_HIP(hipEventRecord(ev_fork_, stream_));
                RV_HIP(hipStreamWaitEvent(stream2_, ev_fork_, 0));
                for (int q = 1; q <= 3; ++q)
                    if (L.n_ot[ob][q] > L.na_ot[ob][q])
                        timed_schur(stream2_, q == 3 ? 0 : q, L.n_ot[ob][q] - L.na_ot[ob][q],
                                    (const TileItem *)D(L.o_ot[ob][q]) + L.na_ot[ob][q], L.dSnap[par], 1, wpp);
                if (L.n_ot[ob][0] > L.na_ot[ob][0])
                    timed_outer(stream2_, L.n_ot[ob][0] - L.na_ot[ob][0],
                                (const TileItem *)D(L.o_ot[ob][0]) + L.na_ot[ob][0], L.dSnap[par], wpp);
                RV_HIP(hipEventRecord(ev_join_, stream2_));
                la_pending = true;
                ++la_launches_;
            }
        }
        if (la_pending) {
            RV_HIP(hipStreamWaitEvent(stream_, ev_join_, 0));
            la_pending = false;
        }
        if (o_.failed_pivot_tpp)
            hipLaunchKernelGGL((k_tpp_left<512, 4>), dim3(std::min(na, TPP_LEFT_WG)), dim3(512), TPP_LDS_MAX, stream_,
                               d_fr_, L.dleft, o_.threshold, o_.small, (unsigned)TPP_LDS_MAX);
    }
    // ---- kept factor columns of the pooled fronts: final from here on, read beside the
    // contribution GEMMs (which only read them) on stream2_, joined after the collect (measured
    // against a copy beside the next level's pivoting, which slows that latency-bound chain
    // more) ----
    const bool kf_fork = L.nkf && !capturing_;
    if (L.nkf) {
        hipStream_t ks = stream_;
        if (kf_fork) {
            ensure_stream2();
            RV_HIP(hipEventRecord(ev_fork_, stream_));
            RV_HIP(hipStreamWaitEvent(stream2_, ev_fork_, 0));
            ks = stream2_;
        }
        hipLaunchKernelGGL(k_keep_factor, dim3((unsigned)L.nkf), dim3(256), 0, ks, (const FrontDev *)d_fr_,
                           (const int2 *)D(L.o_kf));
        if (kf_fork) RV_HIP(hipEventRecord(ev_join_, stream2_));
    }
    // ---- contribution blocks ----
    if (L.nct[0] + L.nct[1] + L.nct[2] + L.nct[3]) {
        hipLaunchKernelGGL(k_form_ld, dim3((unsigned)L.nf0), dim3(256), 0, stream_, d_fr_,
                           (const AptpState *)nullptr, (const int4 *)D(L.o_f0), 0, (double *const *)D(L.o_wp0),
                           (AptpState *)nullptr);
        for (int q = 0; q < 4; ++q)
            if (L.nct[q])
                timed_schur(stream_, q, L.nct[q], (const TileItem *)D(L.o_ct[q]), nullptr, 0, (double *const *)D(L.o_wp0));
    }
    // ---- collect ----
    hipLaunchKernelGGL(k_collect, dim3(nf), dim3(256), 0, stream_, d_fr_, (const int *)D(L.o_ids),
                       (const long long *)D(L.o_doffs), (int *)L.dres, (int *)(L.dres + L.res_del_off));
    if (kf_fork) RV_HIP(hipStreamWaitEvent(stream_, ev_join_, 0));
    L.hres = pin_take(L.res_bytes);
    RV_HIP(hipMemcpyAsync(L.hres, L.dres, L.res_bytes, hipMemcpyDeviceToHost, stream_));
}

void NumericGPU::read_level(int lv) {
    const Prepared &P = *prep_;
    LevelPlan &L = plans_[lv];
    const std::vector<int> &fronts = P.levels[lv];
    const int nf = L.nf;
    const int *hr = (const int *)L.hres;
    const unsigned long long *hml = (const unsigned long long *)(L.hres + (size_t)nf * RES_INTS * sizeof(int));
    const double *huf = (const double *)(hml + nf);
    const int *hdel = (const int *)(L.hres + L.res_del_off);
    for (int li = 0; li < nf; ++li) {
        const int s = fronts[li];
        const int *r = hr + li * RES_INTS;
        if (r[7] & 1) chain_err_ = true;
        if (r[7] & 2) la_err_ = true;
        obfail_[s] = (unsigned long long)(unsigned)r[8] | ((unsigned long long)(unsigned)r[9] << 32);
        ne_[s] = r[0];
        n1_[s] = r[1];
        n2_[s] = r[2];
        zp_[s] = r[3];
        inert_[s][0] = r[4];
        inert_[s][1] = r[5];
        inert_[s][2] = r[6];
        unsigned long long bits = hml[li];
        double v;
        std::memcpy(&v, &bits, sizeof(v));
        maxl_[s] = v;
        h_fr_[s].ne = ne_[s];
        delayed_[s].assign(hdel + L.doffs[li], hdel + L.doffs[li] + (k_[s] - ne_[s]));
    }
    if (!L.sev.empty()) {
        // algorithmic flops: contribution blocks 2 ne nfs(nfs+1)/2, outer updates from k_outer_end
        double fl = 0, flc = 0, maxnfs = 0;
        for (int li = 0; li < nf; ++li) {
            const int s = fronts[li];
            fl += huf[li];
            if (P.sns[s].parent < 0) continue;
            const double nfs = m_[s] - k_[s];
            flc += (double)ne_[s] * nfs * (nfs + 1.0);
            maxnfs = std::max(maxnfs, nfs);
        }
        fl += flc;
        const bool big = maxnfs >= 2048;
        for (size_t q = 0; q < L.sev.size(); ++q) {
            auto &e = L.sev[q];
            float ms = 0.f;
            RV_HIP(hipEventElapsedTime(&ms, e.first, e.second));
            times_.schur_ms += ms;
            times_.schur_launches += 1;
            if (big && q < L.sev_contrib.size() && L.sev_contrib[q]) {
                times_.big_ms += ms;
                times_.big_launches += 1;
            }
            (void)hipEventDestroy(e.first);
            (void)hipEventDestroy(e.second);
        }
        L.sev.clear();
        L.sev_contrib.clear();
        times_.schur_flops += fl;
        if (big) times_.big_flops += flc;
    }
}

#ifdef RV_PHASE_TIMING
}  // namespace rv
extern "C" void rv_debug_phases(double *out) {
    unsigned long long h[2][16], n[2];
    (void)hipMemcpyFromSymbol(h, HIP_SYMBOL(rv::g_phase), sizeof(h));
    (void)hipMemcpyFromSymbol(n, HIP_SYMBOL(rv::g_phase_launches), sizeof(n));
    for (int k = 0; k < 2; ++k)
        for (int i = 0; i < 16; ++i) out[k * 17 + i] = n[k] ? (double)h[k][i] / (double)n[k] : 0.0;
    out[16] = (double)n[0];
    out[33] = (double)n[1];
}
namespace rv {
#endif

bool NumericGPU::front_held(int s) const {
    return pool_block_[s] < 0 || !pool_.clobbered(pool_block_[s]);
}

void NumericGPU::export_raw(int s, double *Fh, int *perm, int *rows) const {
    if (!front_held(s))
        throw std::runtime_error("the working front of supernode " + std::to_string(s) +
                                 " was handed to a later level (RV_KEEP_FRONTS=1 keeps it)");
    const FrontDev &F = h_fr_[s];
    const int m = F.m;
    if (Fh) RV_HIP(hipMemcpy(Fh, F.F, (size_t)m * m * sizeof(double), hipMemcpyDeviceToHost));
    if (perm) RV_HIP(hipMemcpy(perm, F.perm, m * sizeof(int), hipMemcpyDeviceToHost));
    if (rows) RV_HIP(hipMemcpy(rows, F.rows, m * sizeof(int), hipMemcpyDeviceToHost));
}

// Contribution block of front s (ContributionBlock, numeric.rs:516-523): the trailing
// (m - ne) x (m - ne) block of the front after its Schur update, rows [delayed columns in APTP
// order, pattern rows].  Returns its order, 0 for a root or a fully eliminated front.
int NumericGPU::export_contribution(int s, double *data, int *rows, int *num_delayed) const {
    const FrontDev &F = h_fr_[s];
    const int m = F.m, k = F.k, ne = ne_[s];
    const int size = m - ne;
    if (prep_->sns[s].parent < 0 || size <= 0) return 0;
    if (!front_held(s))
        throw std::runtime_error("the contribution block of supernode " + std::to_string(s) +
                                 " was handed to a later level (RV_KEEP_FRONTS=1 keeps it)");
    if (num_delayed) *num_delayed = k - ne;
    if (data)
        RV_HIP(hipMemcpy2D(data, (size_t)size * sizeof(double), F.F + ne + (size_t)ne * m,
                           (size_t)m * sizeof(double), (size_t)size * sizeof(double), size,
                           hipMemcpyDeviceToHost));
    if (rows) {
        std::vector<int> perm(m), r(m);
        RV_HIP(hipMemcpy(perm.data(), F.perm, m * sizeof(int), hipMemcpyDeviceToHost));
        RV_HIP(hipMemcpy(r.data(), F.rows, m * sizeof(int), hipMemcpyDeviceToHost));
        int q = 0;
        for (int i = ne; i < k; ++i) rows[q++] = r[perm[i]];
        for (int i = k; i < m; ++i) rows[q++] = r[i];
    }
    return size;
}

void NumericGPU::front_d(int s, signed char *kind, double *diag, double *off) const {
    const FrontDev &F = h_fr_[s];
    const int ne = ne_[s];
    if (ne == 0) return;
    std::vector<int8_t> kd(ne);
    RV_HIP(hipMemcpy(kd.data(), F.dkind, ne, hipMemcpyDeviceToHost));
    if (diag) RV_HIP(hipMemcpy(diag, F.ddiag, ne * sizeof(double), hipMemcpyDeviceToHost));
    if (off) RV_HIP(hipMemcpy(off, F.doff, ne * sizeof(double), hipMemcpyDeviceToHost));
    for (int c = 0; c < ne; ++c) {
        if (kind) kind[c] = (signed char)(kd[c] == 3 ? 2 : kd[c]);
        if (off && kd[c] != 2) off[c] = 0.0;
    }
}

void NumericGPU::supernode_info(int s, long long out[8], double *max_l) const {
    out[0] = m_[s]; out[1] = k_[s]; out[2] = ne_[s]; out[3] = k_[s] - ne_[s];
    out[4] = n1_[s]; out[5] = n2_[s]; out[6] = prep_->sns[s].parent;
    out[7] = prep_->sns[s].in_small_leaf ? 1 : 0;
    if (max_l) *max_l = maxl_[s];
}

// Features of every front for the update-precision classifier, from the supernode structure and
// the last factorization (16 per front, row-major): sizes, update and front flops, position in the
// tree, assembled contribution volume, delays in and out, 2x2 and negative-pivot fractions,
// largest |L|, and the ratio to the parent's order.
void NumericGPU::front_features(float *out) const {
    const Prepared &P = *prep_;
    const int ns = (int)P.sns.size();
    std::vector<int> lvl(ns, 0);
    const int nl = (int)P.levels.size();
    for (int l = 0; l < nl; ++l)
        for (int s : P.levels[l]) lvl[s] = l;
    auto lg = [](double v) { return (float)std::log2(1.0 + std::max(v, 0.0)); };
    for (int s = 0; s < ns; ++s) {
        const double m = m_[s], k = k_[s], ne = ne_[s], nfs = m - k;
        double din = 0.0, cvol = 0.0;
        for (int c : P.children[s]) {
            din += (double)delayed_[c].size();
            const double sc = m_[c] - ne_[c];
            cvol += sc * sc;
        }
        const double ff = ((m - 1) * m * (m + 1) - (m - k - 1) * (m - k) * (m - k + 1)) / 3.0;
        const int par = P.sns[s].parent;
        float *f = out + (size_t)s * 16;
        f[0] = lg(m);
        f[1] = lg(k);
        f[2] = lg(nfs);
        f[3] = (float)(m > 0 ? k / m : 0.0);
        f[4] = lg(ne * nfs * (nfs + 1));
        f[5] = lg(ff);
        f[6] = (float)(nl > 1 ? (double)lvl[s] / (nl - 1) : 0.0);
        f[7] = lg((double)P.children[s].size());
        f[8] = lg(cvol);
        f[9] = (float)(k > 0 ? din / k : 0.0);
        f[10] = (float)(k > 0 ? (k - ne) / k : 0.0);
        f[11] = (float)(2.0 * n2_[s] / std::max(1.0, ne));
        f[12] = (float)std::log10(1.0 + maxl_[s]);
        f[13] = (float)(inert_[s][1] / std::max(1.0, ne));
        f[14] = par < 0 ? 1.0f : 0.0f;
        f[15] = (float)(par < 0 || m_[par] == 0 ? 0.0 : m / m_[par]);
    }
}

// inertia from the D factors (diagonal.rs:391-461), summed over fronts (solver.rs:504-519)
void NumericGPU::inertia(long long out[3]) const {
    // per-front counts from k_collect; the unresolved delays at the roots are not in D
    out[0] = out[1] = out[2] = 0;
    for (const auto &c : inert_)
        for (int i = 0; i < 3; ++i) out[i] += c[i];
}

void NumericGPU::export_front(int s, double *l11, double *l21, signed char *dkind, double *ddiag,
                              double *doff, int *col_indices, int *row_indices,
                              int *local_perm) const {
    const FrontDev &F = h_fr_[s];
    const int m = F.m, k = F.k, ne = ne_[s];
    std::vector<double> A((size_t)m * std::max(ne, 1));
    if (ne) RV_HIP(hipMemcpy(A.data(), F.Lf, (size_t)m * ne * sizeof(double), hipMemcpyDeviceToHost));
    std::vector<int> perm(m), rows(m);
    RV_HIP(hipMemcpy(perm.data(), F.perm, m * sizeof(int), hipMemcpyDeviceToHost));
    RV_HIP(hipMemcpy(rows.data(), F.rows, m * sizeof(int), hipMemcpyDeviceToHost));
    std::vector<int8_t> kind(std::max(ne, 1));
    std::vector<double> dg(std::max(ne, 1)), of(std::max(ne, 1));
    if (ne) {
        RV_HIP(hipMemcpy(kind.data(), F.dkind, ne, hipMemcpyDeviceToHost));
        RV_HIP(hipMemcpy(dg.data(), F.ddiag, ne * sizeof(double), hipMemcpyDeviceToHost));
        RV_HIP(hipMemcpy(of.data(), F.doff, ne * sizeof(double), hipMemcpyDeviceToHost));
    }
    // extract_front_factors (numeric.rs:2579-2713)
    if (l11) {
        for (int j = 0; j < ne; ++j)
            for (int i = 0; i < ne; ++i) l11[i + (size_t)j * ne] = 0.0;
        int col = 0;
        while (col < ne) {
            l11[col + (size_t)col * ne] = 1.0;
            if (kind[col] == 1) {
                for (int i = col + 1; i < ne; ++i) l11[i + (size_t)col * ne] = A[i + (size_t)col * m];
                col += 1;
            } else {
                l11[(col + 1) + (size_t)(col + 1) * ne] = 1.0;
                for (int i = col + 2; i < ne; ++i) {
                    l11[i + (size_t)col * ne] = A[i + (size_t)col * m];
                    l11[i + (size_t)(col + 1) * ne] = A[i + (size_t)(col + 1) * m];
                }
                col += 2;
            }
        }
    }
    const int r = m - ne;
    if (l21)
        for (int j = 0; j < ne; ++j)
            for (int i = 0; i < r; ++i) l21[i + (size_t)j * r] = A[(ne + i) + (size_t)j * m];
    for (int c = 0; c < ne; ++c) {
        if (dkind) dkind[c] = (signed char)(kind[c] == 3 ? 2 : kind[c]);
        if (ddiag) ddiag[c] = dg[c];
        if (doff) doff[c] = (kind[c] == 2) ? of[c] : 0.0;
        if (col_indices) col_indices[c] = rows[perm[c]];
    }
    if (row_indices) {
        int q = 0;
        for (int i = ne; i < k; ++i) row_indices[q++] = rows[perm[i]];
        for (int i = k; i < m; ++i) row_indices[q++] = rows[i];
    }
    if (local_perm)
        for (int i = 0; i < k; ++i) local_perm[i] = perm[i];
}

}  // namespace rv
