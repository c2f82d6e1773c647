// Triangular solves with LU factors, FP64 residuals and refinement updates.
//
// Replaces LAPACKE_zgetrs ("wersja referencyjna/Wire_MoM.cu":382) and
// cublasZgetrsBatched ("wersja gpu/Wire_MoM.cu":477): B is permuted by the
// pivot sequence, then L y = P b (unit lower) and U x = y are solved.
//
// Each triangular solve is one launch.  Workgroup i owns row block i (64
// rows).  It subtracts the contributions of the blocks already solved, as
// each one becomes ready (its values arrive as tagged packets, written by the
// block's workgroup after its solve), and then solves its diagonal block
// inside one wave with lane broadcasts.  A workgroup only ever waits on
// blocks owned by workgroups with a smaller id in the same grid, which are
// dispatched before it, so the chain always makes progress; every wait is
// bounded.  Arithmetic is FP64; complex64 factors are widened on load.
#include <algorithm>
#include <cfloat>
#include <cstring>
#include <mutex>
#include <vector>

#include "wm_cplx.h"
#include "wm_internal.h"

namespace wm {

namespace {

constexpr int TB = 64;  // rows per block

template <typename T>
__device__ inline double2 ld2(const typename CT<T>::V *p)
{
    const typename CT<T>::V v = *p;
    return make_double2((double)v.x, (double)v.y);
}

// acc -= a*b with every rounding written out (fused multiply-adds), so a
// value does not depend on how the compiler contracts the instantiation it
// is inlined into (the right-hand-side count of a triangular solve).
__device__ inline void cfms(double2 &acc, double2 a, double2 b)
{
    acc.x = fma(-a.x, b.x, acc.x);
    acc.x = fma(a.y, b.y, acc.x);
    acc.y = fma(-a.x, b.y, acc.y);
    acc.y = fma(-a.y, b.x, acc.y);
}

// acc += a*b, roundings written out as in cfms.
__device__ inline void cfma(double2 &acc, double2 a, double2 b)
{
    acc.x = fma(a.x, b.x, acc.x);
    acc.x = fma(-a.y, b.y, acc.x);
    acc.y = fma(a.x, b.y, acc.y);
    acc.y = fma(a.y, b.x, acc.y);
}

// perm[t] = source row of position t after applying ipiv in order: each thread
// follows its position through the interchanges backwards, last to first, so
// the matrix's rows are traced side by side instead of the interchanges applied
// one after another by one thread (N = 8192, two matrices: 0.8 -> 0.36 ms of a
// solve).
__global__ __launch_bounds__(256) void k_perm(const int *ipiv, int64_t strideP, int n, int *perm, int64_t strideQ,
                                              const int *bidx)
{
    const int b = bidx ? bidx[blockIdx.y] : (int)blockIdx.y;
    const int *ip = ipiv + (size_t)b * strideP;
    const int t = blockIdx.x * 256 + threadIdx.x;
    int row = t;
#pragma unroll 16
    for (int i = n - 1; i >= 0; --i) {
        const int p = ip[i] - 1;  // uniform: scalar loads
        row = row == i ? p : row == p ? i : row;
    }
    if (t < n) perm[(size_t)b * strideQ + t] = row;
}

struct TrsvArgs {
    const void *A;
    int lda;
    int64_t strideA;
    int n, nrhs;
    const int *perm;
    int64_t strideQ;
    const double2 *Bin;   // lower solve: right-hand sides (gathered through perm), per launch member
    int ldb;
    int64_t strideB;
    double2 *Y;           // output (lower: y, upper: x in place of y)
    uint64_t *pkt;        // solved values as tagged packets: per member [block][rhs][row][4 words]
    int epoch;            // packet tag of this launch
    int *err;
    const int *bidx;      // launch member -> matrix index of B and Y (null: identity)
    const int *aidx;      // launch member -> matrix index of the factors and permutation (null: as bidx)
};

// Packed entries of one 64 x 64 triangle with its diagonal.
constexpr int kPack = TB * (TB + 1) / 2;

__device__ inline double bcast(double v, int lane)  // value of `lane` to the whole wave
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)(u & 0xffffffffu), lane);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The double whose low and high words lanes `l` and `l + 1` hold, to the whole wave.
__device__ inline double word_pair(uint32_t w, int l)
{
    const unsigned lo = __builtin_amdgcn_readlane(w, l), hi = __builtin_amdgcn_readlane(w, l + 1);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Packed index of element (i, j) of the 64 x 64 diagonal block, column by
// column (so the lanes of a wave, one row each, read consecutive entries of
// a column: no LDS bank conflicts): strictly lower part for L (i > j), upper
// part with the diagonal for U (i <= j).
__device__ inline int dl_idx(int i, int j) { return j * (2 * TB - 1 - j) / 2 + (i - j - 1); }
__device__ inline int du_idx(int i, int j) { return j * (j + 1) / 2 + i; }

// Triangular solve, one launch.  Workgroup (member, g) owns row block bi of
// that launch member (lower: g, upper: nblk-1-g); lower solves L y = P b,
// upper solves U x = y in place, and also publishes each solved value as four
// tagged packets for the later blocks.  The grid is (members, blocks), so
// workgroup ids run over the members first: the resident workgroups hold the
// leading blocks of every member and all members' chains advance together.
// Waits only on blocks of workgroups with smaller ids (dispatched earlier).
//
// TRANS solves with the conjugate transposes of the factors (A^H = U^H L^H P):
// the lower pass takes U^H (lower, non-unit diagonal conj(u_ii)) on the
// right-hand sides as staged (no gather), the upper pass L^H (upper, unit
// diagonal) in place; element (i, j) of the triangle is conj(A(j, i)).  The
// caller scatters the result through the permutation (x = P^T w).
template <typename T, int NR, bool UPPER, bool TRANS>
__global__ __launch_bounds__(256) void k_trsv(TrsvArgs a, int r_off)
{
    // no contraction: a right-hand side's arithmetic is the same in every
    // instantiation (NR), so grouping columns never changes their values
#pragma clang fp contract(off)
    using V = typename CT<T>::V;
    constexpr bool UNIT = TRANS ? UPPER : !UPPER;  // unit diagonal (L or L^H)
    // element (i, j) of the triangle being solved
    auto elem = [&](const V *A, int i, int j) -> double2 {
        if (!TRANS) return ld2<T>(A + i + (size_t)j * a.lda);
        const double2 v = ld2<T>(A + j + (size_t)i * a.lda);
        return make_double2(v.x, -v.y);
    };
    const int bl = blockIdx.x, tid = threadIdx.x, row = tid & 63;
    const int b = a.bidx ? a.bidx[bl] : bl;
    const int fb = a.aidx ? a.aidx[bl] : b;  // factors (and their permutation) of this member
    const int part = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nblk = a.n / TB;
    const int bi = UPPER ? nblk - 1 - (int)blockIdx.y : (int)blockIdx.y, r0 = bi * TB;
    const V *A = (const V *)a.A + (size_t)fb * a.strideA;
    double2 *Y = a.Y + (size_t)b * a.strideB + (size_t)r_off * a.ldb;
    uint64_t *pk = a.pkt + (size_t)bl * nblk * NR * 256;
    const uint32_t tag = (uint32_t)a.epoch;
    const int nr = a.nrhs - r_off;

    // diagonal block to LDS (independent of other blocks, so before any wait)
    constexpr int kPad = 1;  // dl_idx(0, 0) is -1
    __shared__ double2 s_d[kPad + kPack];
    __shared__ double2 s_rd[TB];
    for (int e = tid; e < TB * TB; e += 256) {
        // consecutive threads walk down a column of the stored factor
        const int i = TRANS ? e / TB : e % TB, j = TRANS ? e % TB : e / TB;
        if (!UPPER && i > j) s_d[kPad + dl_idx(i, j)] = elem(A, r0 + i, r0 + j);
        if (UPPER && i < j) s_d[kPad + du_idx(i, j)] = elem(A, r0 + i, r0 + j);
        if (!UNIT && i == j) {
            const double2 u = elem(A, r0 + i, r0 + j);
            s_rd[i] = crecip(u.x, u.y);
        }
    }

    double2 acc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = make_double2(0.0, 0.0);
    if (part == 0) {
        const int src = (UPPER || TRANS) ? r0 + row : a.perm[(size_t)fb * a.strideQ + r0 + row];
        const double2 *in = UPPER ? Y : a.Bin + (size_t)bl * a.strideB + (size_t)r_off * a.ldb;
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (r < nr) acc[r] = in[src + (size_t)r * a.ldb];
    }

    // off-diagonal blocks in dependency order, next block prefetched
    const int nb_off = UPPER ? nblk - 1 - bi : bi;
    auto blk = [&](int q) { return UPPER ? nblk - 1 - q : q; };
    double2 lcur[16], lnext[16];
    if (nb_off > 0) {
        const int c0 = blk(0) * TB + part * 16;
#pragma unroll
        for (int c = 0; c < 16; ++c) lcur[c] = elem(A, r0 + row, c0 + c);
    }
    for (int q = 0; q < nb_off; ++q) {
        // The part's 16 solved values of block q: 64 packets per right-hand
        // side, one per lane, polled until the block's workgroup has tagged
        // them (a value and its readiness in one memory round trip), and all
        // loaded before the next block's L prefetch.
        const uint64_t *pq = pk + (size_t)blk(q) * NR * 256 + part * 64 + row;
        uint32_t yw[NR];
        long it = 0;
        for (;;) {
            bool got = true;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                yw[r] = 0u;
                if (r < nr) {
                    const uint64_t v = ld_pkt(pq + r * 256);
                    yw[r] = (uint32_t)v;
                    got = got && (uint32_t)(v >> 32) == tag;
                }
            }
            if (__all(got)) break;
            if (spin_give_up(it, a.err)) break;
        }
        __builtin_amdgcn_sched_barrier(0);
        if (q + 1 < nb_off) {
            const int c1 = blk(q + 1) * TB + part * 16;
#pragma unroll
            for (int c = 0; c < 16; ++c) lnext[c] = elem(A, r0 + row, c1 + c);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 16; ++c) {
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (r < nr) cfms(acc[r], lcur[c], make_double2(word_pair(yw[r], 4 * c), word_pair(yw[r], 4 * c + 2)));
        }
#pragma unroll
        for (int c = 0; c < 16; ++c) lcur[c] = lnext[c];
    }

    // The four parts' sums meet in LDS; wave p then solves the right-hand
    // sides p, p + 4, ... (each sum in the order part 0 + 1 + 2 + 3, so a
    // value does not depend on NR or on which wave solves it).
    __shared__ double2 s_acc[4][TB][NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) s_acc[part][row][r] = acc[r];
    __syncthreads();
    constexpr int RW = (NR + 3) / 4;  // right-hand sides per wave
    if (part < NR) {
        double2 x[RW];
#pragma unroll
        for (int k = 0; k < RW; ++k) {
            const int r = part + 4 * k;
            x[k] = make_double2(0.0, 0.0);
            if (r < NR) {
                x[k] = s_acc[0][row][r];
#pragma unroll
                for (int p = 1; p < 4; ++p) { x[k].x += s_acc[p][row][r].x; x[k].y += s_acc[p][row][r].y; }
            }
        }
        // The substitution is the launch's critical path: unrolled, and without
        // branches.  A step broadcasts row j's value (every lane scales it by the
        // diagonal's reciprocal), and the rows that it reaches take the
        // difference by selection: the others read some entry of the packed
        // block and drop the product, so a step's LDS reads need no mask and
        // are issued ahead of it.
#pragma unroll
        for (int jj = 0; jj < TB; ++jj) {
            const int j = UPPER ? TB - 1 - jj : jj;
            const double2 l = s_d[kPad + (UPPER ? du_idx(row, j) : dl_idx(row, j))];
            const double2 ri = UNIT ? make_double2(1.0, 0.0) : s_rd[j];
#pragma unroll
            for (int k = 0; k < RW; ++k) {
                if (part + 4 * k >= NR) break;
                double2 xj = make_double2(bcast(x[k].x, j), bcast(x[k].y, j));
                if (!UNIT) xj = make_double2(xj.x * ri.x - xj.y * ri.y, xj.x * ri.y + xj.y * ri.x);
                double2 v = x[k];
                cfms(v, l, xj);
                const bool below = UPPER ? row < j : row > j;
                x[k].x = below ? v.x : !UNIT && row == j ? xj.x : x[k].x;
                x[k].y = below ? v.y : !UNIT && row == j ? xj.y : x[k].y;
            }
        }
#pragma unroll
        for (int k = 0; k < RW; ++k) {
            const int r = part + 4 * k;
            if (r < nr) {
                Y[(r0 + row) + (size_t)r * a.ldb] = x[k];
                uint64_t *pw = pk + ((size_t)bi * NR + r) * 256 + row * 4;
                const uint64_t xb = (uint64_t)__double_as_longlong(x[k].x), yb = (uint64_t)__double_as_longlong(x[k].y);
                put_pkt(pw, tag, (uint32_t)xb);
                put_pkt(pw + 1, tag, (uint32_t)(xb >> 32));
                put_pkt(pw + 2, tag, (uint32_t)yb);
                put_pkt(pw + 3, tag, (uint32_t)(yb >> 32));
            }
        }
    }
}

// Partial products P[split][row][r] = sum_{j in split} Z[row][j] X[j][r].
// Lane = row (each column of Z is one coalesced 1 KiB read per wave); the
// wave's column range is wave-uniform, so X arrives through scalar loads.  Z
// streams through in batches of kZB columns (all loads of a batch issued
// before its products, non-temporal: Z is read once per product), and each
// column's term is added in column order with fused multiply-adds, so a
// row's sum depends on n only.
typedef double d2v __attribute__((ext_vector_type(2)));

// ABS: also the split's partial row sums of |Z| (the infinity norm of Z, taken
// in the same pass over Z), Pabs[(member * nsplit + split) * n + row].
template <int NR, bool ABS>
__global__ __launch_bounds__(256) void k_resid_part(const double2 *Z, int ldz, int64_t strideZ, int n, int nrhs,
                                                    const double2 *X, int ldb, int64_t strideB, int cols_per_split,
                                                    int nsplit, double2 *P, int r_off, const int *bidx, double *Pabs)
{
    constexpr int kZB = 8;
    const int bl = blockIdx.z, split = blockIdx.y, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b = bidx ? bidx[bl] : bl;
    const int row = blockIdx.x * 64 + lane;
    const double2 *Zb = Z + (size_t)b * strideZ;
    const double2 *Xb = X + (size_t)b * strideB + (size_t)r_off * ldb;
    const int cw = cols_per_split / 4;
    const int c0 = split * cols_per_split + wave * cw;
    // NR <= nrhs - r_off: the launcher runs right-hand sides in chunks of 8, 4, 2, 1
    double2 acc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = make_double2(0.0, 0.0);
    double asum = 0.0;
    const double2 *zp = Zb + row + (size_t)c0 * ldz;
    for (int c = 0; c < cw; c += kZB) {  // cw is a multiple of kZB
        double2 z[kZB];
#pragma unroll
        for (int e = 0; e < kZB; ++e) {
            const d2v v = __builtin_nontemporal_load((const d2v *)(zp + (size_t)(c + e) * ldz));
            z[e] = make_double2(v.x, v.y);
        }
#pragma unroll
        for (int e = 0; e < kZB; ++e) {
#pragma unroll
            for (int r = 0; r < NR; ++r) cfma(acc[r], z[e], Xb[c0 + c + e + (size_t)r * ldb]);
            if (ABS) asum += hypot(z[e].x, z[e].y);
        }
    }
    __shared__ double2 s[3][64][NR];
    __shared__ double sa[3][64];
    if (wave > 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r) s[wave - 1][lane][r] = acc[r];
        if (ABS) sa[wave - 1][lane] = asum;
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
#pragma unroll
            for (int p = 0; p < 3; ++p) { acc[r].x += s[p][lane][r].x; acc[r].y += s[p][lane][r].y; }
            P[(((size_t)bl * nsplit + split) * NR + r) * n + row] = acc[r];
        }
        if (ABS) {
#pragma unroll
            for (int p = 0; p < 3; ++p) asum += sa[p][lane];
            Pabs[((size_t)bl * nsplit + split) * n + row] = asum;
        }
    }
}

// R = B - sum_split P, in split order.  With Pabs: the row sums of |Z| (in
// split order) over the leading np rows, their maximum into znorm[b] as the
// ordered bit pattern of a non-negative double (non-finite as +inf).
template <int NR>
__global__ void k_resid_final(const double2 *P, int nsplit, int n, int nrhs, const double2 *B, int ldb,
                              int64_t strideB, double2 *R, int r_off, const int *bidx, const double *Pabs, int np,
                              unsigned long long *znorm)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int bl = blockIdx.y;
    const int b = bidx ? bidx[bl] : bl;
    if (Pabs) {  // uniform per launch
        double a = 0.0;
        if (i < np) {
            for (int sp = 0; sp < nsplit; ++sp) a += Pabs[((size_t)bl * nsplit + sp) * n + i];
            if (!(a <= DBL_MAX)) a = INFINITY;
        }
        for (int off = 32; off >= 1; off >>= 1) a = fmax(a, __shfl_xor(a, off));
        if ((threadIdx.x & 63) == 0) atomicMax(&znorm[b], (unsigned long long)__double_as_longlong(a));
    }
    if (i >= n) return;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        if (r >= nrhs - r_off) break;
        double2 s = make_double2(0.0, 0.0);
        for (int sp = 0; sp < nsplit; ++sp) {
            const double2 p = P[(((size_t)bl * nsplit + sp) * NR + r) * n + i];
            s.x += p.x;
            s.y += p.y;
        }
        const size_t o = (size_t)b * strideB + (size_t)(r_off + r) * ldb + i;
        R[o] = B ? make_double2(B[o].x - s.x, B[o].y - s.y) : s;  // no B: the product Z X
    }
}

template <typename T, int NR, bool TRANS>
void launch_trsv(const TrsvArgs &a, int batch, int r_off, bool upper, hipStream_t s)
{
    const dim3 grid(batch, a.n / TB);
    if (upper) hipLaunchKernelGGL((k_trsv<T, NR, true, TRANS>), grid, dim3(256), 0, s, a, r_off);
    else hipLaunchKernelGGL((k_trsv<T, NR, false, TRANS>), grid, dim3(256), 0, s, a, r_off);
}

// Inverses of the 64 x 64 diagonal blocks of LU factors, FP64 arithmetic:
// blockIdx = (block, triangle 0 = L (unit lower) / 1 = U, slot); slot z
// takes the factors of index fidx[z].  Lane j solves for column j of the
// inverse by substitution against the block staged in LDS; the inverse is
// stored whole, column by column, zeros in its other triangle.
template <typename T>
__global__ __launch_bounds__(64) void k_diag_inv(const void *F, int lda, int64_t strideF, const int *fidx, int nblk,
                                                 double2 *Dinv)
{
#pragma clang fp contract(off)
    using V = typename CT<T>::V;
    const int bi = blockIdx.x, upper = blockIdx.y, j = threadIdx.x, r0 = bi * TB;
    const V *A = (const V *)F + (size_t)fidx[blockIdx.z] * strideF;
    __shared__ double2 s_t[TB][TB + 1];  // the block, s_t[i][k] = A(r0 + i, r0 + k)
    __shared__ double2 s_x[TB][TB + 1];  // the inverse, column j by lane j
    for (int e = j; e < TB * TB; e += TB) {
        const int i = e % TB, k = e / TB;
        s_t[i][k] = ld2<T>(A + (r0 + i) + (size_t)(r0 + k) * lda);
    }
    __syncthreads();
    if (!upper) {
        for (int i = 0; i < TB; ++i) {
            double2 v = make_double2(i == j ? 1.0 : 0.0, 0.0);
            if (i > j)
                for (int k = j; k < i; ++k) cfms(v, s_t[i][k], s_x[k][j]);
            s_x[i][j] = v;
        }
    } else {
        for (int i = TB - 1; i >= 0; --i) {
            double2 v = make_double2(i == j ? 1.0 : 0.0, 0.0);
            if (i <= j) {
                for (int k = i + 1; k <= j; ++k) cfms(v, s_t[i][k], s_x[k][j]);
                const double2 d = s_t[i][i], rd = crecip(d.x, d.y);
                v = make_double2(v.x * rd.x - v.y * rd.y, v.x * rd.y + v.y * rd.x);
            }
            s_x[i][j] = v;
        }
    }
    __syncthreads();
    double2 *D = Dinv + (((size_t)blockIdx.z * 2 + upper) * nblk + bi) * TB * TB;
    for (int e = j; e < TB * TB; e += TB) {
        const int i = e % TB, k = e / TB;
        D[e] = (upper ? i <= k : i >= k) ? s_x[i][k] : make_double2(0.0, 0.0);
    }
}

typedef double v4d __attribute__((ext_vector_type(4)));

// Preconditioner factors: every row block of L and U times the inverse of its
// diagonal block, L' = diag(L_ii)^-1 L and U' = diag(U_ii)^-1 U, so that a solve
// needs no work on the diagonal between one block's values and the next's.
// blockIdx = (column block, row block, slot); row block bi of factor fidx[z],
// column block cb (left of the diagonal: L, right of it: U) is multiplied by
// its inverse on the matrix cores (three real products per complex product,
// lanes as in k_psolve) and written to dst, which may be the factors themselves.
template <typename T>
__global__ __launch_bounds__(256) void k_scale_blocks(const void *F, double2 *dst, int lda, int64_t strideF,
                                                      const int *fidx, int nblk, const double2 *Dinv)
{
    using V = typename CT<T>::V;
    const int cb = blockIdx.x, bi = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (cb == bi) return;
    const int upper = cb > bi;
    const size_t base = (size_t)fidx[blockIdx.z] * strideF + (size_t)bi * TB + (size_t)cb * TB * lda;
    const V *A = (const V *)F + base;
    const double2 *D = Dinv + (((size_t)blockIdx.z * 2 + upper) * nblk + bi) * TB * TB;
    __shared__ double2 s_t[TB][TB];  // s_t[k][(column + k) % TB]: both sides free of bank conflicts
    for (int e = tid; e < TB * TB; e += 256) {
        // consecutive lanes walk down a column
        s_t[e % TB][(e / TB + e % TB) % TB] = ld2<T>(A + e % TB + (size_t)(e / TB) * lda);
    }
    __syncthreads();
    v4d P[4], Q[4], S[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) P[c] = Q[c] = S[c] = v4d{0, 0, 0, 0};
    for (int k = lane / 16; k < TB; k += 4) {
        const double2 d = D[(size_t)k * TB + wave * 16 + lane % 16];
        const double ds = d.x + d.y;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const double2 t = s_t[k][(c * 16 + lane % 16 + k) % TB];
            P[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x, d.x, P[c], 0, 0, 0);
            Q[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.y, d.y, Q[c], 0, 0, 0);
            S[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(t.x + t.y, ds, S[c], 0, 0, 0);
        }
    }
    double2 *O = dst + base + wave * 16 + lane % 16;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            O[(size_t)(c * 16 + lane / 16 + 4 * v) * lda] =
                make_double2(P[c][v] - Q[c][v], S[c][v] - P[c][v] - Q[c][v]);
}

// Preconditioner solve L' y = diag(L_ii)^-1 P b (UPPER: U' x = diag(U_ii)^-1 y) for up
// to kPsW right-hand sides per launch member, one launch.  Workgroup (member,
// g) owns row block bi (lower: g, upper: nblk-1-g): c = D_ii^-1 b, then c minus
// the products with the solved blocks as their values arrive, on the matrix
// cores (wave w < 4: rows 16 w ..; three real products per complex product; a
// right-hand side is a column of the products, so its values do not depend on
// its neighbours).  Values of a block travel as plain 8-byte words: a member's
// blocks are filled with kPsEmpty, a NaN pattern no arithmetic produces, before
// the launch, and a reader polls its words until they hold something else.
// Four more waves do the polling: a wave's loads complete in order, so a poll
// behind the next block's factor entries would wait for HBM in every step.
// Waits only on blocks of workgroups with smaller ids (dispatched earlier).
//
// What bounds it: the chain of n / 64 blocks, 2.0 us each with up to 4 columns and
// 3.6 us with 16 (0.5 us for the values to cross, the rest the product of the
// newest block: 48 4x4x4 products per wave for 4 columns, 96 for 8, 48 16x16x4,
// at four times the cycles each, above).  The 4x4x4 form spends nothing on
// columns that are not there and rounds like the 16x16x4 one: a column has the
// same bits in every width.  Per triangle at N = 8192, against substitution by
// inverted diagonal blocks on the vector units, four columns per member:
//   1 factor, 3 columns    258 us instead of 1004
//   2 factors, 16 columns  466 us instead of 1245 (factors read once, not 4 times)
//   N = 512, 3 columns      18 us instead of 65
// One polling wave instead of four: 470 us for 1 x 3 before the 4x4x4 form, 355
// with four; real and imaginary words apart (whole lines per store): 470 us
// instead of 628 for 2 x 16.
constexpr int kPsW = 16;
constexpr int kPsPoll = 4;
constexpr uint64_t kPsEmpty = 0x7ff8b10c5e7afe55ull;

struct PsolveArgs {
    const double2 *F;       // scaled factors
    int lda;
    int64_t strideF;
    int n;
    const double2 *dinv;
    const double *in;       // right-hand sides, [member][block][kPsW][re, im][TB]
    uint64_t *pub;          // solved values, the same layout
    const int *fac, *slot, *width;  // per member: factor, its slot in dinv, its right-hand sides
    int *err;
};

template <bool UPPER>
__global__ __launch_bounds__(256 + 64 * kPsPoll) void k_psolve(PsolveArgs a)
{
    const int bl = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nblk = a.n / TB;
    const int bi = UPPER ? nblk - 1 - (int)blockIdx.y : (int)blockIdx.y, r0 = bi * TB;
    const int w = a.width[bl];
    uint64_t *pub = a.pub + (size_t)bl * a.n * kPsW * 2;
    const int noff = UPPER ? nblk - 1 - bi : bi;
    auto blk = [&](int q) { return UPPER ? nblk - 1 - q : q; };
    // two buffers: a block's values are staged while the previous ones are read
    __shared__ double2 s_y[2][kPsW][TB + 1];

    if (wave >= 4) {  // the values of the other blocks: lane = row, wave 4 + j has columns j, j + kPsPoll, ...
        constexpr int kE = kPsW / kPsPoll;
        const int j0 = wave - 4;
        __syncthreads();
        for (int q = 0; q < noff; ++q) {
            const uint64_t *py = pub + (((size_t)blk(q) * kPsW + j0) * 2) * TB + lane;
            uint64_t yx[kE], yy[kE];
            long it = 0;
            for (;;) {
#pragma unroll
                for (int e = 0; e < kE; ++e) {
                    yx[e] = yy[e] = 0;
                    if (j0 + kPsPoll * e < w) {
                        yx[e] = ld_pkt(py + 2 * kPsPoll * TB * e);
                        yy[e] = ld_pkt(py + 2 * kPsPoll * TB * e + TB);
                    }
                }
                bool got = true;
#pragma unroll
                for (int e = 0; e < kE; ++e) got = got & (yx[e] != kPsEmpty) & (yy[e] != kPsEmpty);
                if (__all(got)) break;
                if (spin_give_up(it, a.err)) break;
            }
#pragma unroll
            for (int e = 0; e < kE; ++e)
                if (j0 + kPsPoll * e < w)
                    s_y[(q + 1) & 1][j0 + kPsPoll * e][lane] = make_double2(
                        __longlong_as_double((long long)yx[e]), __longlong_as_double((long long)yy[e]));
            __syncthreads();
        }
        return;
    }

    const double2 *A = a.F + (size_t)a.fac[bl] * a.strideF;
    const double2 *D = a.dinv + (((size_t)a.slot[bl] * 2 + (UPPER ? 1 : 0)) * nblk + bi) * TB * TB;
    const int row = wave * 16 + lane % 16, kq = lane / 16, rhs = lane % 16;
    double2 lcur[16], lnext[16];  // this lane's factor entries: row, columns kq + 4 t of a block
    auto load_block = [&](int q, double2 *l) {
        const double2 *p = A + r0 + row + (size_t)(q * TB + kq) * a.lda;
#pragma unroll
        for (int t = 0; t < 16; ++t) l[t] = p[(size_t)(4 * t) * a.lda];
    };
    v4d P, Q, S;
    auto product = [&](const double2 *l, int buf) {
        P = Q = S = v4d{0, 0, 0, 0};
        if (w <= 4) {
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const double2 y = s_y[buf][lane % 4][4 * t + kq];
                P[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x, l[t].x, P[0], 0, 0, 0);
                Q[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.y, l[t].y, Q[0], 0, 0, 0);
                S[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x + y.y, l[t].x + l[t].y, S[0], 0, 0, 0);
            }
            return;
        }
        if (w <= 8) {
#pragma unroll
            for (int t = 0; t < 16; ++t) {
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const double2 y = s_y[buf][4 * g + lane % 4][4 * t + kq];
                    P[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x, l[t].x, P[g], 0, 0, 0);
                    Q[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.y, l[t].y, Q[g], 0, 0, 0);
                    S[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x + y.y, l[t].x + l[t].y, S[g], 0, 0, 0);
                }
            }
            return;
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const double2 y = s_y[buf][rhs][4 * t + kq];
            P = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, l[t].x, P, 0, 0, 0);
            Q = __builtin_amdgcn_mfma_f64_16x16x4f64(y.y, l[t].y, Q, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x + y.y, l[t].x + l[t].y, S, 0, 0, 0);
        }
    };

    // c = D^-1 b (this lane: row `row`, right-hand sides kq + 4 v)
    const double *in = a.in + (((size_t)bl * nblk + bi) * kPsW + wave) * 2 * TB + lane;
#pragma unroll
    for (int e = 0; e < 4; ++e) s_y[0][wave + 4 * e][lane] = make_double2(in[8 * TB * e], in[8 * TB * e + TB]);
#pragma unroll
    for (int t = 0; t < 16; ++t) lcur[t] = D[row + (size_t)(4 * t + kq) * TB];
    __syncthreads();
    product(lcur, 0);
    double cr[4], ci[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        cr[v] = P[v] - Q[v];
        ci[v] = S[v] - P[v] - Q[v];
    }
    auto subtract = [&]() {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            cr[v] -= P[v] - Q[v];
            ci[v] -= S[v] - P[v] - Q[v];
        }
    };
    // Two blocks per turn, loads without a condition (past the end: the last
    // block once more), so that a product's wait counts leave the next block's
    // loads in flight; an odd block goes first.
    int q = noff & 1;
    if (q) {
        load_block(blk(0), lnext);
        load_block(blk(min(1, noff - 1)), lcur);
        __syncthreads();
        product(lnext, 1);
        subtract();
    } else if (noff > 0) {
        load_block(blk(0), lcur);
    }
    for (; q < noff; q += 2) {
        load_block(blk(q + 1), lnext);
        __syncthreads();
        product(lcur, (q + 1) & 1);
        subtract();
        load_block(blk(min(q + 2, noff - 1)), lcur);
        __syncthreads();
        product(lnext, q & 1);
        subtract();
    }
    auto word = [](double x) {
        const uint64_t u = (uint64_t)__double_as_longlong(x);
        return u == kPsEmpty ? 0x7ff8000000000000ull : u;
    };
    uint64_t *o = pub + (size_t)bi * kPsW * 2 * TB + row;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (kq + 4 * v < w) {
            uint64_t *ov = o + (kq + 4 * v) * 2 * TB;
            __hip_atomic_store(ov, word(cr[v]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(ov + TB, word(ci[v]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
}

// Right-hand sides of a preconditioner solve, [member][block][kPsW][re, im][TB]:
// rows through perm of column cols[member * kPsW + j] of V (element offset; -1:
// zero), and both triangles' values marked empty (pub, pub + members * n *
// kPsW complex words).
__global__ void k_ps_gather(const double2 *V, int n, const int64_t *cols, const int *fac, const int *perm,
                            int64_t strideQ, double *in, uint64_t *pub, int members)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x, m = blockIdx.y;
    if (t >= n * kPsW) return;
    const int row = t / (TB * kPsW) * TB + t % TB, j = t / TB % kPsW;
    const int64_t c = cols[(size_t)m * kPsW + j];
    const size_t o = (size_t)m * n * kPsW * 2 + (size_t)(t / TB) * 2 * TB + t % TB;
    const double2 v = c >= 0 ? V[c + perm[(size_t)fac[m] * strideQ + row]] : make_double2(0.0, 0.0);
    in[o] = v.x;
    in[o + TB] = v.y;
    const size_t half = (size_t)members * n * kPsW * 2;
    pub[o] = pub[o + TB] = pub[half + o] = pub[half + o + TB] = kPsEmpty;
}

// The solved columns back to V.
__global__ void k_ps_scatter(const double *pub, int n, const int64_t *cols, double2 *V)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x, m = blockIdx.y;
    if (t >= n * kPsW) return;
    const int row = t / (TB * kPsW) * TB + t % TB, j = t / TB % kPsW;
    const int64_t c = cols[(size_t)m * kPsW + j];
    const double *p = pub + (size_t)m * n * kPsW * 2 + (size_t)(t / TB) * 2 * TB + t % TB;
    if (c >= 0) V[c + row] = make_double2(p[0], p[TB]);
}

// Right-hand sides handled by one pass starting at r_off: 8, 4, 2 or 1.
inline int rhs_chunk(int left) { return left >= 8 ? 8 : left >= 4 ? 4 : left >= 2 ? 2 : 1; }

template <typename T, bool TRANS = false>
void trsv_dispatch(const TrsvArgs &a, int batch, int r_off, bool upper, hipStream_t s)
{
    switch (rhs_chunk(a.nrhs - r_off)) {
        case 8: launch_trsv<T, 8, TRANS>(a, batch, r_off, upper, s); break;
        case 4: launch_trsv<T, 4, TRANS>(a, batch, r_off, upper, s); break;
        case 2: launch_trsv<T, 2, TRANS>(a, batch, r_off, upper, s); break;
        default: launch_trsv<T, 1, TRANS>(a, batch, r_off, upper, s); break;
    }
}

// Bstage[member] = B[matrix] (n x nrhs columns with leading dimension ldb)
__global__ void k_stage(const double2 *B, int ldb, int64_t strideB, int n, int nrhs, double2 *S, const int *bidx)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, bl = blockIdx.y;
    const int b = bidx ? bidx[bl] : bl;
    if (i >= n) return;
    for (int r = 0; r < nrhs; ++r) S[(size_t)bl * strideB + (size_t)r * ldb + i] = B[(size_t)b * strideB + (size_t)r * ldb + i];
}

// S[member][perm[t]] = B[matrix][t] (the scatter x = P^T w of a transposed solve)
__global__ void k_unperm(const double2 *B, int ldb, int64_t strideB, int n, int nrhs, const int *perm,
                         int64_t strideQ, double2 *S, const int *bidx, const int *aidx)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, bl = blockIdx.y;
    const int b = bidx ? bidx[bl] : bl;
    if (i >= n) return;
    const int t = perm[(size_t)(aidx ? aidx[bl] : b) * strideQ + i];
    for (int r = 0; r < nrhs; ++r) S[(size_t)bl * strideB + (size_t)r * ldb + t] = B[(size_t)b * strideB + (size_t)r * ldb + i];
}

// B[matrix] = S[member]
__global__ void k_unstage(const double2 *S, int ldb, int64_t strideB, int n, int nrhs, double2 *B, const int *bidx)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, bl = blockIdx.y;
    const int b = bidx ? bidx[bl] : bl;
    if (i >= n) return;
    for (int r = 0; r < nrhs; ++r) B[(size_t)b * strideB + (size_t)r * ldb + i] = S[(size_t)bl * strideB + (size_t)r * ldb + i];
}

__global__ void k_zero_words(int *p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

}  // namespace

int perm_batched(wm_ctx *ctx, int n, const int *ipiv, int64_t strideP, int *perm, int64_t strideQ, int batch,
                 hipStream_t s, const int *d_bidx)
{
    if ((size_t)n * sizeof(int) > ctx->max_lds) {  // the accepted range of n (40960 rows)
        set_error("permutation: n=%d exceeds the LDS capacity", n);
        return WM_ERR_ARG;
    }
    hipLaunchKernelGGL(k_perm, dim3((unsigned)((n + 255) / 256), (unsigned)batch), dim3(256), 0, s, ipiv, strideP, n, perm, strideQ, d_bidx);
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

namespace {

// Buffers of a triangular solve supplied by the caller instead of the
// context's (the allocation-free entry point): staging of B (batch * strideB
// complex128) and the packets of both triangles, zeroed by the caller, whose
// epochs then start at 1.
struct SolveBufs {
    double2 *stage = nullptr;
    uint64_t *pkt = nullptr;
    int epoch = 0;
};

// Packets of the two triangles of a batched solve.
size_t solve_pkts(int n, int nrhs, int batch) { return 2 * (size_t)batch * (n / TB) * rhs_chunk(nrhs) * 256; }

// Staging of B per launch member in ctx->ws_solve; the solved values'
// packets in ctx->ws_pkt, per triangle and member nblk x NR x 256 packets.
// trans: solve A^H X = B instead of A X = B.  ext: caller-supplied buffers
// (nothing allocated, no profiler events).
int getrs_any(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA, const int *perm,
              int64_t strideQ, void *B, int ldb, int64_t strideB, int batch, hipStream_t s, const int *d_bidx,
              bool trans, const int *d_aidx, SolveBufs *ext = nullptr)
{
    if (n <= 0 || n % TB != 0 || nrhs <= 0 || batch <= 0 || ldb < n) {
        set_error("getrs: bad arguments (n=%d multiple of %d, nrhs=%d, batch=%d)", n, TB, nrhs, batch);
        return WM_ERR_ARG;
    }
    const int nblk = n / TB;
    const int nr_max = rhs_chunk(nrhs);
    const size_t tri_pkts = (size_t)batch * nblk * nr_max * 256;  // packets per triangle
    double2 *Ystage = nullptr;
    uint64_t *pkt = nullptr;
    int *epoch = nullptr;
    if (ext) {
        Ystage = ext->stage;
        pkt = ext->pkt;
        epoch = &ext->epoch;
    } else {
        WM_TRY(ctx->ws_solve.ensure((size_t)batch * strideB * sizeof(double2)));
        Ystage = (double2 *)ctx->ws_solve.ptr;
        // The packets live in their own buffer and only ever carry epoch tags of
        // this context, so a wait can never be satisfied by stale data.  The
        // buffer is zeroed whenever it is (re)allocated.
        const size_t pkt_bytes = 2 * tri_pkts * sizeof(uint64_t);
        if (ctx->ws_pkt.bytes < pkt_bytes || !ctx->ws_pkt.ptr) {
            WM_TRY(ctx->ws_pkt.ensure(pkt_bytes));
            const int64_t nf = (int64_t)(ctx->ws_pkt.bytes / sizeof(int));
            hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, s, (int *)ctx->ws_pkt.ptr, nf);
            ctx->solve_epoch = 0;
        }
        pkt = (uint64_t *)ctx->ws_pkt.ptr;
        if (ctx->solve_epoch > (1 << 30)) {  // keep the tags unique: restart from a zeroed buffer
            const int64_t nf = (int64_t)(ctx->ws_pkt.bytes / sizeof(int));
            hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, s, (int *)pkt, nf);
            ctx->solve_epoch = 0;
        }
        epoch = &ctx->solve_epoch;
    }
    // the lower solve reads B (staged per member) and writes y into B; the upper solves in place
    hipLaunchKernelGGL(k_stage, dim3((n + 255) / 256, batch), dim3(256), 0, s, (const double2 *)B, ldb, strideB, n, nrhs,
                       Ystage, d_bidx);
    for (int r0 = 0; r0 < nrhs; r0 += rhs_chunk(nrhs - r0)) {
        TrsvArgs a;
        a.A = A; a.lda = lda; a.strideA = strideA; a.n = n; a.nrhs = nrhs;
        a.perm = perm; a.strideQ = strideQ; a.ldb = ldb; a.strideB = strideB; a.err = ctx->d_err;
        a.bidx = d_bidx;
        a.aidx = d_aidx;
        a.Bin = Ystage; a.Y = (double2 *)B; a.pkt = pkt;
        a.epoch = ++*epoch;
        const int nr = rhs_chunk(nrhs - r0);
        const double esz = prec == WM_PREC_F64 ? 16.0 : 8.0;
        const double fl = batch * 4.0 * (double)n * n * nr, by = batch * 0.5 * (double)n * n * esz;
        for (int up = 0; up < 2; ++up) {
            if (up) { a.Bin = nullptr; a.pkt = pkt + tri_pkts; }
            if (!ext) prof_begin(ctx, K_TRSV, s);
            if (prec == WM_PREC_F64) {
                if (trans) trsv_dispatch<double, true>(a, batch, r0, up, s);
                else trsv_dispatch<double>(a, batch, r0, up, s);
            } else {
                if (trans) trsv_dispatch<float, true>(a, batch, r0, up, s);
                else trsv_dispatch<float>(a, batch, r0, up, s);
            }
            if (!ext) prof_end(ctx, K_TRSV, s, fl, by);
        }
    }
    if (trans) {  // x = P^T w, through the staging buffer
        hipLaunchKernelGGL(k_unperm, dim3((n + 255) / 256, batch), dim3(256), 0, s, (const double2 *)B, ldb, strideB, n,
                           nrhs, perm, strideQ, Ystage, d_bidx, d_aidx);
        hipLaunchKernelGGL(k_unstage, dim3((n + 255) / 256, batch), dim3(256), 0, s, (const double2 *)Ystage, ldb,
                           strideB, n, nrhs, (double2 *)B, d_bidx);
    }
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

}  // namespace

int getrs_perm_batched(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA,
                       const int *perm, int64_t strideQ, void *B, int ldb, int64_t strideB, int batch, hipStream_t s,
                       const int *d_bidx, const int *d_aidx)
{
    return getrs_any(ctx, prec, n, nrhs, A, lda, strideA, perm, strideQ, B, ldb, strideB, batch, s, d_bidx, false,
                     d_aidx);
}

int getrsh_perm_batched(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA,
                        const int *perm, int64_t strideQ, void *B, int ldb, int64_t strideB, int batch, hipStream_t s,
                        const int *d_bidx)
{
    return getrs_any(ctx, prec, n, nrhs, A, lda, strideA, perm, strideQ, B, ldb, strideB, batch, s, d_bidx, true,
                     nullptr);
}

namespace {

// S[member * W + j] = column cols[member * W + j] of V (element offset; -1: zeros).
__global__ void k_gather_cols(const double2 *V, int n, const int64_t *cols, double2 *S)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, mj = blockIdx.y;
    if (i >= n) return;
    const int64_t c = cols[mj];
    S[(size_t)mj * n + i] = c >= 0 ? V[c + i] : make_double2(0.0, 0.0);
}

// The columns back: V[cols[member * W + j]] = S[member * W + j].
__global__ void k_scatter_cols(const double2 *S, int n, const int64_t *cols, double2 *V)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, mj = blockIdx.y;
    if (i >= n) return;
    const int64_t c = cols[mj];
    if (c >= 0) V[c + i] = S[(size_t)mj * n + i];
}

}  // namespace

size_t precond_bytes(int n, int nfac) { return (size_t)nfac * 2 * n * TB * sizeof(double2); }

int precond_prepare(wm_ctx *ctx, int prec, int n, const void *F, int lda, int64_t strideF,
                    const std::vector<int> &factors, double2 *Fs, double2 *Dinv, hipStream_t s)
{
    if (factors.empty()) return WM_OK;
    if (n % TB != 0) {
        set_error("precond_prepare: n=%d not a multiple of %d", n, TB);
        return WM_ERR_ARG;
    }
    WM_TRY(ctx->ws_dinv_idx.ensure(factors.size() * sizeof(int)));
    WM_TRY(copy_h2d(ctx->ws_dinv_idx.ptr, factors.data(), factors.size() * sizeof(int), s));
    const unsigned nblk = (unsigned)(n / TB), nf = (unsigned)factors.size();
    const int *fidx = (const int *)ctx->ws_dinv_idx.ptr;
    if (prec == WM_PREC_F64) {
        hipLaunchKernelGGL(k_diag_inv<double>, dim3(nblk, 2, nf), dim3(TB), 0, s, F, lda, strideF, fidx, n / TB, Dinv);
        hipLaunchKernelGGL(k_scale_blocks<double>, dim3(nblk, nblk, nf), dim3(256), 0, s, F, Fs, lda, strideF, fidx,
                           n / TB, (const double2 *)Dinv);
    } else {
        hipLaunchKernelGGL(k_diag_inv<float>, dim3(nblk, 2, nf), dim3(TB), 0, s, F, lda, strideF, fidx, n / TB, Dinv);
        hipLaunchKernelGGL(k_scale_blocks<float>, dim3(nblk, nblk, nf), dim3(256), 0, s, F, Fs, lda, strideF, fidx,
                           n / TB, (const double2 *)Dinv);
    }
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

namespace {

// Columns of items that share a factor, cut into members of up to max_w: the
// factor of each member and W column offsets (-1: none) per member.
int group_columns(int n, int nr, int64_t strideV, const std::vector<int> &items, const std::vector<int> &fac,
                  int max_w, std::vector<int> &member_fac, std::vector<int64_t> &cols, int &W)
{
    // the columns of each factor, factors in the order of their first item
    std::vector<int> order;
    std::vector<std::vector<int64_t>> cols_of;
    std::vector<int> pos_of;  // factor index -> position in order (grown on demand)
    for (size_t q = 0; q < items.size(); ++q) {
        const int f = fac[q];
        if (f < 0) {
            set_error("grouped solve: item %d has no factors", items[q]);
            return WM_ERR_ARG;
        }
        if ((size_t)f >= pos_of.size()) pos_of.resize((size_t)f + 1, -1);
        if (pos_of[f] < 0) {
            pos_of[f] = (int)order.size();
            order.push_back(f);
            cols_of.emplace_back();
        }
        for (int r = 0; r < nr; ++r) cols_of[pos_of[f]].push_back((int64_t)items[q] * strideV + (int64_t)r * n);
    }
    size_t widest = 0;
    for (const auto &c : cols_of) widest = std::max(widest, c.size());
    W = 1;  // right-hand sides per launch member: a power of two, at most max_w
    while (W < max_w && (size_t)W < widest) W *= 2;
    if (max_w == kPsW) W = kPsW;
    for (size_t g = 0; g < order.size(); ++g)
        for (size_t j0 = 0; j0 < cols_of[g].size(); j0 += W) {
            member_fac.push_back(order[g]);
            for (int j = 0; j < W; ++j)
                cols.push_back(j0 + j < cols_of[g].size() ? cols_of[g][j0 + j] : (int64_t)-1);
        }
    return WM_OK;
}

}  // namespace

int precond_solve(wm_ctx *ctx, int n, int nr, const double2 *Fs, int lda, int64_t strideF, const int *perm,
                  int64_t strideQ, const double2 *Dinv, const std::vector<int> &slot_of, double2 *V, int64_t strideV,
                  const std::vector<int> &items, const std::vector<int> &fac, hipStream_t s)
{
    if (items.empty()) return WM_OK;
    if (items.size() != fac.size() || nr <= 0 || strideV < (int64_t)n * nr || n % TB != 0) {
        set_error("precond_solve: bad arguments");
        return WM_ERR_ARG;
    }
    std::vector<int> mf;
    std::vector<int64_t> cols;
    int W = kPsW;
    WM_TRY(group_columns(n, nr, strideV, items, fac, kPsW, mf, cols, W));
    const int members = (int)mf.size();
    // tables: factor, slot, width per member, then the columns
    std::vector<int> tab(3 * (size_t)members);
    for (int m = 0; m < members; ++m) {
        const int f = mf[m];
        if (f >= (int)slot_of.size() || slot_of[f] < 0) {
            set_error("precond_solve: factor %d was not prepared", f);
            return WM_ERR_ARG;
        }
        tab[m] = f;
        tab[members + m] = slot_of[f];
        int w = 0;
        while (w < kPsW && cols[(size_t)m * kPsW + w] >= 0) ++w;
        tab[2 * members + m] = w;
    }
    const size_t tab_b = (tab.size() * sizeof(int) + 255) & ~(size_t)255;
    const size_t cols_b = (cols.size() * sizeof(int64_t) + 255) & ~(size_t)255;
    const size_t vec_b = (size_t)members * n * kPsW * sizeof(double2);
    WM_TRY(ctx->ws_group.ensure(tab_b + cols_b + 3 * vec_b));
    char *base = (char *)ctx->ws_group.ptr;
    std::vector<char> host(tab_b + cols_b, 0);
    std::memcpy(host.data(), tab.data(), tab.size() * sizeof(int));
    std::memcpy(host.data() + tab_b, cols.data(), cols.size() * sizeof(int64_t));
    WM_TRY(copy_h2d(base, host.data(), host.size(), s));
    const int *d_tab = (const int *)base;
    const int64_t *d_cols = (const int64_t *)(base + tab_b);
    double *in = (double *)(base + tab_b + cols_b);
    uint64_t *pub = (uint64_t *)(base + tab_b + cols_b + vec_b);
    uint64_t *pub2 = pub + (size_t)members * n * kPsW * 2;
    const dim3 grid((unsigned)members, (unsigned)(n / TB)), vgrid((unsigned)(n * kPsW / 256), (unsigned)members);
    const double fl = 4.0 * (double)n * n * items.size() * nr, by = members * 8.0 * (double)n * n;
    hipLaunchKernelGGL(k_ps_gather, vgrid, dim3(256), 0, s,
                       (const double2 *)V, n, d_cols, d_tab, perm, strideQ, in, pub, members);
    PsolveArgs a;
    a.F = Fs; a.lda = lda; a.strideF = strideF; a.n = n; a.dinv = Dinv;
    a.fac = d_tab; a.slot = d_tab + members; a.width = d_tab + 2 * members;
    a.err = ctx->d_err;
    a.in = in; a.pub = pub;
    prof_begin(ctx, K_TRSV, s);
    hipLaunchKernelGGL(k_psolve<false>, grid, dim3(256 + 64 * kPsPoll), 0, s, a);
    prof_end(ctx, K_TRSV, s, fl, by);
    a.in = (const double *)pub; a.pub = pub2;  // the lower triangle's values are the upper one's right-hand sides
    prof_begin(ctx, K_TRSV, s);
    hipLaunchKernelGGL(k_psolve<true>, grid, dim3(256 + 64 * kPsPoll), 0, s, a);
    prof_end(ctx, K_TRSV, s, fl, by);
    hipLaunchKernelGGL(k_ps_scatter, vgrid, dim3(256), 0, s,
                       (const double *)pub2, n, d_cols, V);
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

int getrs_grouped(wm_ctx *ctx, int prec, int n, int nr, const void *F, int lda, int64_t strideF, const int *perm,
                  int64_t strideQ, double2 *V, int64_t strideV, const std::vector<int> &items,
                  const std::vector<int> &fac, hipStream_t s, int max_w)
{
    if (items.empty()) return WM_OK;
    if (items.size() != fac.size() || nr <= 0 || strideV < (int64_t)n * nr) {
        set_error("getrs_grouped: bad arguments");
        return WM_ERR_ARG;
    }
    std::vector<int> aidx;
    std::vector<int64_t> cols;
    int W = 1;
    WM_TRY(group_columns(n, nr, strideV, items, fac, std::min(max_w, 8), aidx, cols, W));
    const int members = (int)aidx.size();
    const size_t aidx_b = ((size_t)members * sizeof(int) + 255) & ~(size_t)255;
    const size_t cols_b = ((size_t)members * W * sizeof(int64_t) + 255) & ~(size_t)255;
    const size_t stage_b = (size_t)members * W * n * sizeof(double2);
    WM_TRY(ctx->ws_group.ensure(aidx_b + cols_b + stage_b));
    char *base = (char *)ctx->ws_group.ptr;
    std::vector<char> host(aidx_b + cols_b, 0);
    std::memcpy(host.data(), aidx.data(), aidx.size() * sizeof(int));
    std::memcpy(host.data() + aidx_b, cols.data(), cols.size() * sizeof(int64_t));
    WM_TRY(copy_h2d(base, host.data(), host.size(), s));
    const int *d_aidx = (const int *)base;
    const int64_t *d_cols = (const int64_t *)(base + aidx_b);
    double2 *S = (double2 *)(base + aidx_b + cols_b);
    const dim3 grid((unsigned)((n + 255) / 256), (unsigned)(members * W));
    hipLaunchKernelGGL(k_gather_cols, grid, dim3(256), 0, s, (const double2 *)V, n, d_cols, S);
    WM_TRY(getrs_any(ctx, prec, n, W, F, lda, strideF, perm, strideQ, S, n, (int64_t)W * n, members, s, nullptr,
                     false, d_aidx));
    hipLaunchKernelGGL(k_scatter_cols, grid, dim3(256), 0, s, (const double2 *)S, n, d_cols, V);
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

int getrs_batched(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA, const int *ipiv,
                  int64_t strideP, void *B, int ldb, int64_t strideB, int batch, hipStream_t s)
{
    WM_TRY(ctx->ws_perm.ensure((size_t)batch * n * sizeof(int)));
    int *perm = (int *)ctx->ws_perm.ptr;
    WM_TRY(perm_batched(ctx, n, ipiv, strideP, perm, n, batch, s));
    return getrs_perm_batched(ctx, prec, n, nrhs, A, lda, strideA, perm, n, B, ldb, strideB, batch, s);
}

int residual_batched(wm_ctx *ctx, int n, int nrhs, const void *Z, int ldz, int64_t strideZ, const void *X,
                     const void *B, int ldb, int64_t strideB, void *R, int batch, hipStream_t s, const int *d_bidx,
                     unsigned long long *znorm, int np)
{
    if (n % 64 != 0) {
        set_error("residual: n=%d not a multiple of 64", n);
        return WM_ERR_ARG;
    }
    // column splits depend on n only, so an item's rounding never depends on the batch
    int nsplit = 1;
    while (nsplit < 16 && n % (nsplit * 2 * 64) == 0 && n / (nsplit * 2) >= 256) nsplit *= 2;
    const int cps = n / nsplit;
    const int nrp = nrhs >= 8 ? 8 : nrhs >= 4 ? 4 : nrhs >= 2 ? 2 : 1;
    DevBuf &partial = ctx->ws_resid;
    const size_t pbytes = (size_t)batch * nsplit * nrp * n * sizeof(double2);
    const size_t need = pbytes + (znorm ? (size_t)batch * nsplit * n * sizeof(double) : 0);
    WM_TRY(partial.ensure(need));
    double *pabs = znorm ? (double *)((char *)partial.ptr + pbytes) : nullptr;
    for (int r0 = 0; r0 < nrhs; r0 += rhs_chunk(nrhs - r0)) {
        const int left = rhs_chunk(nrhs - r0);
        const dim3 g1(n / 64, nsplit, batch), g2((n + 255) / 256, batch);
        // the norm of Z rides along the first right-hand-side chunk only
        double *pa = r0 == 0 ? pabs : nullptr;
#define WM_RESID(NR)                                                                                          \
    if (pa)                                                                                                   \
        hipLaunchKernelGGL((k_resid_part<NR, true>), g1, dim3(256), 0, s, (const double2 *)Z, ldz, strideZ, n, \
                           nrhs, (const double2 *)X, ldb, strideB, cps, nsplit, (double2 *)partial.ptr, r0,     \
                           d_bidx, pa);                                                                       \
    else                                                                                                      \
        hipLaunchKernelGGL((k_resid_part<NR, false>), g1, dim3(256), 0, s, (const double2 *)Z, ldz, strideZ, n, \
                           nrhs, (const double2 *)X, ldb, strideB, cps, nsplit, (double2 *)partial.ptr, r0,     \
                           d_bidx, (double *)nullptr);                                                         \
    hipLaunchKernelGGL(k_resid_final<NR>, g2, dim3(256), 0, s, (const double2 *)partial.ptr, nsplit, n, nrhs,   \
                       (const double2 *)B, ldb, strideB, (double2 *)R, r0, d_bidx, (const double *)pa, np, znorm)
        prof_begin(ctx, K_RESID, s);
        if (left == 8) { WM_RESID(8); }
        else if (left == 4) { WM_RESID(4); }
        else if (left == 2) { WM_RESID(2); }
        else { WM_RESID(1); }
        prof_end(ctx, K_RESID, s, batch * 8.0 * (double)n * n * left, batch * 16.0 * (double)n * n);
#undef WM_RESID
    }
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

}  // namespace wm

// ---------------------------------------------------------------------------
// Allocation-free triangular solves: the staging, permutation and packet
// buffers of wm_getrs_batched live in `scratch`, a file-scope device array of
// kNoAllocBytes that every GPU the library runs on holds until the process
// ends.  Its device address is taken once per device (wm::noalloc_init, from
// wm_init with that device current); host code uses that address, never the
// array's name.  Calls on one GPU share the array: overlapping calls race.
namespace {
constexpr size_t kNoAllocBytes = (size_t)32 << 20;
constexpr int kNoAllocDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];
void *g_scratch_dev[kNoAllocDevices] = {};
std::mutex g_scratch_mu;
}  // namespace

namespace wm {

int noalloc_init(int device)
{
    if (device < 0 || device >= kNoAllocDevices) {
        set_error("scratch: device %d beyond %d", device, kNoAllocDevices);
        return WM_ERR_ARG;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_dev[device]) return WM_OK;
    void *p = nullptr;
    WM_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_dev[device] = p;
    return WM_OK;
}

}  // namespace wm

extern "C" int wm_getrs_batched_noalloc(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda,
                                        int64_t strideA, const int *ipiv, int64_t strideP, wm_c128 *B, int ldb,
                                        int64_t strideB, int batch)
{
    using namespace wm;
    if (!ctx || !A || !ipiv || !B || n <= 0 || n % TB != 0 || nrhs <= 0 || batch <= 0 || ldb < n || lda < n ||
        strideB < (int64_t)ldb * nrhs || (prec != WM_PREC_F64 && prec != WM_PREC_F32 && prec != WM_PREC_BF16X3)) {
        set_error("wm_getrs_batched_noalloc: bad arguments (n=%d a multiple of %d, nrhs=%d, batch=%d, ldb=%d, "
                  "strideB=%lld)", n, TB, nrhs, batch, ldb, (long long)strideB);
        return WM_ERR_ARG;
    }
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t perm_b = up((size_t)batch * n * sizeof(int));
    const size_t stage_b = up((size_t)batch * strideB * sizeof(double2));
    const size_t pkt_b = up(solve_pkts(n, nrhs, batch) * sizeof(uint64_t));
    if (perm_b + stage_b + pkt_b > kNoAllocBytes) {
        set_error("wm_getrs_batched_noalloc: n=%d, nrhs=%d, batch=%d need %zu bytes of scratch, the maximum is %zu "
                  "(use wm_getrs_batched)", n, nrhs, batch, perm_b + stage_b + pkt_b, kNoAllocBytes);
        return WM_ERR_NOMEM;
    }
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    char *base = (char *)g_scratch_dev[ctx->device];
    if (!base) {
        set_error("wm_getrs_batched_noalloc: no scratch address for device %d", ctx->device);
        return WM_ERR_STATE;
    }
    const hipStream_t s = ctx->stream;
    int *perm = (int *)base;
    SolveBufs sb;
    sb.stage = (double2 *)(base + perm_b);
    sb.pkt = (uint64_t *)(base + perm_b + stage_b);
    // the previous call's packets carry the same epochs: start from zero
    const int64_t nw = (int64_t)(pkt_b / sizeof(int));
    hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s, (int *)sb.pkt, nw);
    WM_TRY(perm_batched(ctx, n, ipiv, strideP, perm, n, batch, s));
    WM_TRY(getrs_any(ctx, prec, n, nrhs, A, lda, strideA, perm, n, B, ldb, strideB, batch, s, nullptr, false, nullptr,
                     &sb));
    return check_device_error(ctx, s);
}

// Internal test hook (not part of include/wiremom.h): grouped solves.  Item q
// (vectors at V + items[q] * strideV, nr columns of n) is solved in place with
// the factors fac[q] of wm_getrf_batched (device buffers, stride n * n; pivots
// stride n).
extern "C" int wmx_getrs_grouped(wm_ctx *ctx, int prec, int n, int nr, const void *A, int nfac, const int *ipiv,
                                 wm_c128 *V, int64_t strideV, int nitems, const int *items, const int *fac, int inv,
                                 int max_w)
{
    using namespace wm;
    if (!ctx || !A || !ipiv || !V || nitems <= 0 || nfac <= 0) {
        set_error("wmx_getrs_grouped: bad arguments");
        return WM_ERR_ARG;
    }
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    WM_TRY(ctx->ws_perm.ensure((size_t)nfac * n * sizeof(int)));
    int *perm = (int *)ctx->ws_perm.ptr;
    WM_TRY(perm_batched(ctx, n, ipiv, n, perm, n, nfac, ctx->stream));
    const std::vector<int> its(items, items + nitems), fs(fac, fac + nitems);
    if (!inv) {
        WM_TRY(getrs_grouped(ctx, prec, n, nr, A, n, (int64_t)n * n, perm, n, (double2 *)V, strideV, its, fs,
                             ctx->stream, max_w > 0 ? max_w : 8));
        return check_device_error(ctx, ctx->stream);
    }
    // the preconditioner's solves, on a scaled copy of the factors
    std::vector<int> slot(nfac);
    for (int f = 0; f < nfac; ++f) slot[f] = f;
    WM_TRY(ctx->ws_dinv.ensure(precond_bytes(n, nfac)));
    double2 *dinv = (double2 *)ctx->ws_dinv.ptr, *copy = nullptr;
    WM_HIP_TRY(hipMalloc(&copy, (size_t)nfac * n * n * sizeof(double2)));
    int rc = precond_prepare(ctx, prec, n, A, n, (int64_t)n * n, slot, copy, dinv, ctx->stream);
    if (rc == WM_OK)
        rc = precond_solve(ctx, n, nr, copy, n, (int64_t)n * n, perm, n, dinv, slot, (double2 *)V, strideV, its, fs,
                           ctx->stream);
    if (rc == WM_OK) rc = check_device_error(ctx, ctx->stream);
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipFree(copy);
    return rc;
}

// Internal test hook (not part of include/wiremom.h): solves A^H X = B with the
// factors and pivots of wm_getrf_batched (device buffers, as wm_getrs_batched).
extern "C" int wmx_getrs_trans(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA,
                               const int *ipiv, int64_t strideP, wm_c128 *B, int ldb, int64_t strideB, int batch)
{
    using namespace wm;
    if (!ctx || !A || !ipiv || !B || batch <= 0) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    WM_TRY(ctx->ws_perm.ensure((size_t)batch * n * sizeof(int)));
    int *perm = (int *)ctx->ws_perm.ptr;
    WM_TRY(perm_batched(ctx, n, ipiv, strideP, perm, n, batch, ctx->stream));
    WM_TRY(getrsh_perm_batched(ctx, prec, n, nrhs, A, lda, strideA, perm, n, B, ldb, strideB, batch, ctx->stream));
    WM_HIP_TRY(hipStreamSynchronize(ctx->stream));
    return check_device_error(ctx, ctx->stream);
}
