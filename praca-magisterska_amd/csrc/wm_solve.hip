// Triangular solves with LU factors, FP64 residuals and refinement updates.
//
// Replaces LAPACKE_zgetrs ("wersja referencyjna/Wire_MoM.cu":382) and
// cublasZgetrsBatched ("wersja gpu/Wire_MoM.cu":477): B is permuted by the
// pivot sequence, then L y = P b (unit lower) and U x = y are solved.
//
// Each triangular solve is one launch.  Workgroup i owns row block i (64
// rows).  It subtracts the contributions of the blocks already solved, as
// each one becomes ready (its values arrive in words that were marked empty
// before, written by the block's workgroup after its solve), and then solves
// its diagonal block, a column per wave, with lane broadcasts.  A workgroup only ever waits on
// blocks owned by workgroups with a smaller id in the same grid, which are
// dispatched before it, so the chain always makes progress; every wait is
// bounded.  Arithmetic is FP64; complex64 factors are widened on load.
#include <algorithm>
#include <cfloat>
#include <cstring>
#include <mutex>
#include <type_traits>
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

// Source row of position t after applying ipiv in order: each thread follows
// its position through the interchanges backwards, last to first.  A thread's
// trace is a serial chain (35 cycles per interchange: the pivots of 64 of them in
// one load, a lane read each), so a long sequence is cut into kPermParts parts
// traced side by side (blockIdx.y; map[member][part][position]) and the parts'
// maps are followed one through the other (k_perm_join).  N = 8192, two
// matrices: 50 us; one thread swapping in LDS 800, one part 470 (with scalar loads).
constexpr int kPermParts = 8;
constexpr int kPermWhole = 512;  // up to here one part: the join costs more than it saves

__global__ __launch_bounds__(256) void k_perm(const int *ipiv, int64_t strideP, int n, int len, int *out,
                                              int64_t strideOut, const int *bidx, int map)
{
    const int bl = blockIdx.z, part = blockIdx.y, lane = threadIdx.x & 63;
    const int b = bidx ? bidx[bl] : bl;
    const int *ip = ipiv + (size_t)b * strideP;
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int i_lo = part * len, i_hi = min(n, i_lo + len);  // len is a multiple of 64
    auto load = [&](int i0) { return i0 + lane < i_hi ? ip[i0 + lane] - 1 : i0 + lane; };
    int row = t;
    int i0 = i_lo + (i_hi - i_lo - 1) / 64 * 64;
    int next = load(i0);
    for (; i0 >= i_lo; i0 -= 64) {
        const int cur = next;
        if (i0 > i_lo) next = load(i0 - 64);
#pragma unroll
        for (int k = 63; k >= 0; --k) {
            const int p = __builtin_amdgcn_readlane(cur, k), i = i0 + k;
            row = row == i ? p : row == p ? i : row;
        }
    }
    if (t < n) out[(map ? (size_t)bl * kPermParts + part : (size_t)b) * strideOut + t] = row;
}

__global__ __launch_bounds__(256) void k_perm_join(const int *map, int n, int *perm, int64_t strideQ, const int *bidx)
{
    const int bl = blockIdx.y, t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    int row = t;
    for (int part = kPermParts - 1; part >= 0; --part) {
        if ((unsigned)row >= (unsigned)n) break;  // a pivot outside the matrix
        row = map[((size_t)bl * kPermParts + part) * n + row];
    }
    perm[(size_t)(bidx ? bidx[bl] : bl) * strideQ + t] = row;
}

// Packed entries of one 64 x 64 triangle with its diagonal.
constexpr int kPack = TB * (TB + 1) / 2;

__device__ inline double bcast(double v, int lane)  // value of `lane` to the whole wave
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)(u & 0xffffffffu), lane);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Packed index of element (i, j) of the 64 x 64 diagonal block, column by
// column (so the lanes of a wave, one row each, read consecutive entries of
// a column: no LDS bank conflicts): strictly lower part for L (i > j), upper
// part with the diagonal for U (i <= j).
__device__ inline int dl_idx(int i, int j) { return j * (2 * TB - 1 - j) / 2 + (i - j - 1); }
__device__ inline int du_idx(int i, int j) { return j * (j + 1) / 2 + i; }

typedef double v4d __attribute__((ext_vector_type(4)));

// Right-hand sides in one pass of a triangular solve: kPsW per launch member
// (columns of the matrix products), kPassCols per matrix.
constexpr int kPsW = 16;
constexpr int kPassCols = 32;
constexpr int kPsPoll = 4;  // polling waves
constexpr uint64_t kPsEmpty = 0x7ff8b10c5e7afe55ull;

// Values of a pass are kept as [item][block][column][re, im][TB].
struct TrsvArgs {
    const void *A;
    int lda;
    int64_t strideA;
    int n;
    int ncols;         // columns per item
    int chunks;        // launch members per item: member m has columns m % chunks * cw ... of item m / chunks
    int cw;
    const int *bidx;   // item -> matrix (null: identity)
    const int *aidx;   // item -> factors (null: as bidx)
    const int *width;  // SCALED: item -> its columns in use
    const double2 *dinv;  // SCALED: inverted diagonal blocks
    const int *slot;      // SCALED: item -> its factors' blocks in dinv
    uint64_t *in;      // right-hand sides; the lower solve leaves them marked empty, for the upper solve's values
    uint64_t *pub;     // solved values
    int *err;
};

// Triangular solve, one launch.  Workgroup (member, g) owns row block bi of
// that launch member (lower: g, upper: nblk-1-g); lower solves L y = P b,
// upper solves U x = y.  The grid is (members, blocks), so workgroup ids run
// over the members first: the resident workgroups hold the leading blocks of
// every member and all members' chains advance together.  Waits only on blocks
// of workgroups with smaller ids (dispatched earlier).
//
// Four waves (wave w: rows 16 w ..) subtract the products with the solved blocks
// as their values arrive, on the matrix cores; a right-hand side is a column of
// the products, so its values do not depend on its neighbours, and the 4x4x4
// form (up to 8 columns) rounds like the 16x16x4 one.  Then all eight waves
// substitute through the diagonal block, a column each.  Values of a block
// travel as plain 8-byte words: they are marked empty (kPsEmpty, a NaN pattern
// no arithmetic produces) before the launch, and a reader polls its words until
// they hold something else.  The other four waves do the polling: a wave's
// loads complete in order, so a poll behind the next block's factor entries
// would wait for HBM in every step.
//
// TRANS solves with the conjugate transposes of the factors (A^H = U^H L^H P):
// the lower pass takes U^H (lower, non-unit diagonal conj(u_ii)) on the
// right-hand sides as they are (no gather), the upper pass L^H (upper, unit
// diagonal); element (i, j) of the triangle is conj(A(j, i)).  The results
// leave through the permutation (x = P^T w).
//
// SCALED solves with factors whose row blocks are multiplied by the inverses of
// their diagonal blocks (k_scale_blocks): c = D_ii^-1 b at the start instead of
// the substitution, and three real products per complex product instead of
// four.  For preconditioners.
//
// What bounds it: the chain of n / 64 blocks.  SCALED: 2.0 us each with up to 4
// columns and 3.6 us with 16 (0.5 us for the values to cross, the rest the
// product of the newest block: 48 4x4x4 products per wave for 4 columns, 96 for
// 8, 48 16x16x4, at four times the cycles each, above).  Per triangle at N =
// 8192, against substitution by inverted diagonal blocks on the vector units,
// four columns per member:
//   1 factor, 3 columns    258 us instead of 1004
//   2 factors, 16 columns  466 us instead of 1245 (factors read once, not 4 times)
//   N = 512, 3 columns      18 us instead of 65
// One polling wave instead of four: 470 us for 1 x 3 before the 4x4x4 form, 355
// with four; real and imaginary words apart (whole lines per store): 470 us
// instead of 628 for 2 x 16.
// Not SCALED: 5.5 us a block lower and 7.4 us upper with 8 columns in two matrices of
// N = 8192, of which the substitution is about 2.3 and 4 us (76 and 110 cycles a
// step) and the product 1; 827 us per triangle on average instead of 1977 with the
// poll, the products (values broadcast by lane reads) and the substitution of two
// columns per wave in the same four waves, eight columns at most per pass.
//
// SHORT solves matrices of at most two blocks: one product at most and no block
// loaded ahead, so that two workgroups fit on a CU.  A batch of such matrices has no
// chain to wait for, only as many blocks as matrices: 1000 x 64 29 -> 20 us per
// triangle, 300 x 128 27.5 -> 19 (one column; 46 and 42 before the diagonal block's
// loads were issued together).
//
// Otherwise eight waves are two per SIMD, and a third would be another workgroup's:
// the scheduler is told so, or it shortens the distance of the complex64 form's
// loads for an occupancy that no launch has (2 x 8192, eight columns: 904 us instead
// of 852 per triangle).
template <typename T, bool UPPER, bool TRANS, bool SCALED, bool SHORT>
__global__ __launch_bounds__(256 + 64 * kPsPoll)
__attribute__((amdgpu_waves_per_eu(SHORT ? 4 : 2, SHORT ? 4 : 2))) void k_trsv(TrsvArgs a)
{
    // no contraction: a right-hand side's arithmetic is the same in every form
#pragma clang fp contract(off)
    using V = typename CT<T>::V;
    constexpr bool UNIT = TRANS ? UPPER : !UPPER;  // unit diagonal (L or L^H)
    const int item = blockIdx.x / a.chunks, c0 = blockIdx.x % a.chunks * a.cw;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nblk = a.n / TB;
    const int bi = UPPER ? nblk - 1 - (int)blockIdx.y : (int)blockIdx.y, r0 = bi * TB;
    const int w = SCALED ? a.width[item] : min(a.cw, a.ncols - c0);
    const int fb = a.aidx ? a.aidx[item] : a.bidx ? a.bidx[item] : item;
    const V *A = (const V *)a.A + (size_t)fb * a.strideA;
    const double2 *D = a.dinv;
    if (SCALED) D += (((size_t)a.slot[item] * 2 + (UPPER ? 1 : 0)) * nblk + bi) * TB * TB;
    // this member's columns of block q of the item's values
    auto cols_of = [&](uint64_t *v, int q) { return v + (((size_t)item * nblk + q) * a.ncols + c0) * 2 * TB; };
    auto elem = [&](int i, int j) -> double2 {  // element (i, j) of the triangle being solved
        if (!TRANS) return ld2<T>(A + i + (size_t)j * a.lda);
        const double2 v = ld2<T>(A + j + (size_t)i * a.lda);
        return make_double2(v.x, -v.y);
    };
    auto put = [](uint64_t *o, double x) {
        const uint64_t u = (uint64_t)__double_as_longlong(x);
        __hip_atomic_store(o, u == kPsEmpty ? 0x7ff8000000000000ull : u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const int noff = UPPER ? nblk - 1 - bi : bi;
    auto blk = [&](int q) { return UPPER ? nblk - 1 - q : q; };
    // two buffers: a block's values are staged while the previous ones are read
    __shared__ double2 s_y[2][kPsW][TB + 1];
    constexpr int kPad = 1;  // dl_idx(0, 0) is -1
    __shared__ double2 s_d[SCALED ? 1 : kPad + kPack];
    __shared__ double2 s_rd[SCALED ? 1 : TB];

    if (wave >= 4) {
        if (!SCALED) {
            // The whole block in loads without conditions, then the triangle of it to
            // LDS, and the diagonal's reciprocals a lane each.  The blocks that start a
            // chain wait for this (a load under its condition at a time and a reciprocal
            // per column: 11.5 us per triangle of one block instead of 8).
            constexpr int kEl = TB / kPsPoll;
            V v[kEl];
            const V *p = A + r0 + lane + (size_t)(r0 + wave - 4) * a.lda;  // down a column of the stored factor
#pragma unroll
            for (int q = 0; q < kEl; ++q) v[q] = p[(size_t)(kPsPoll * q) * a.lda];
            if (!UNIT && wave == 4) {
                const double2 u = elem(r0 + lane, r0 + lane);
                s_rd[lane] = crecip(u.x, u.y);
            }
#pragma unroll
            for (int q = 0; q < kEl; ++q) {
                const int col = wave - 4 + kPsPoll * q, i = TRANS ? col : lane, j = TRANS ? lane : col;
                const double2 x = make_double2((double)v[q].x, TRANS ? -(double)v[q].y : (double)v[q].y);
                if (!UPPER && i > j) s_d[kPad + dl_idx(i, j)] = x;
                if (UPPER && i < j) s_d[kPad + du_idx(i, j)] = x;
            }
        } else {
            __syncthreads();  // the right-hand sides are staged
        }
        // the values of the other blocks: lane = row, wave 4 + j has columns j, j + kPsPoll, ...
        constexpr int kE = kPsW / kPsPoll;
        const int j0 = wave - 4;
        for (int q = 0; q < noff; ++q) {
            const uint64_t *py = cols_of(a.pub, blk(q)) + j0 * 2 * TB + lane;
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
        if (SCALED) return;
    } else {
        const int row = wave * 16 + lane % 16, kq = lane / 16, rhs = lane % 16;
        V lcur[16], lnext[16];  // this lane's factor entries: row, columns kq + 4 t of a block
        auto load_block = [&](int q, V *l) {
            const size_t step = TRANS ? 1 : (size_t)a.lda;
            const V *p = TRANS ? A + (size_t)(r0 + row) * a.lda + q * TB + kq
                               : A + r0 + row + (size_t)(q * TB + kq) * a.lda;
#pragma unroll
            for (int t = 0; t < 16; ++t) l[t] = p[4 * t * step];
        };
        // P + i R: the products of a block; SCALED: P, Q = re re, im im and R = (re + im)(re + im)
        v4d P, Q, R;
        auto product = [&](const V *l, int buf) {
            P = Q = R = v4d{0, 0, 0, 0};
            auto steps = [&](auto ng_c, auto mul) {
                constexpr int NG = decltype(ng_c)::value;
#pragma unroll
                for (int t = 0; t < 16; ++t) {
                    const double lx = l[t].x, ly = TRANS ? -l[t].y : l[t].y;
#pragma unroll
                    for (int g = 0; g < NG; ++g) mul(t, g, lx, ly);
                }
            };
            auto small = [&](int t, int g, double lx, double ly) {
                const double2 y = s_y[buf][4 * g + lane % 4][4 * t + kq];
                if (SCALED) {
                    P[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x, lx, P[g], 0, 0, 0);
                    Q[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.y, ly, Q[g], 0, 0, 0);
                    R[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x + y.y, lx + ly, R[g], 0, 0, 0);
                } else {
                    P[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x, lx, P[g], 0, 0, 0);
                    R[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.y, lx, R[g], 0, 0, 0);
                    P[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(-y.y, ly, P[g], 0, 0, 0);
                    R[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(y.x, ly, R[g], 0, 0, 0);
                }
            };
            if (w <= 4) {
                steps(std::integral_constant<int, 1>{}, small);
                return;
            }
            if (w <= 8) {
                steps(std::integral_constant<int, 2>{}, small);
                return;
            }
            steps(std::integral_constant<int, 1>{}, [&](int t, int, double lx, double ly) {
                const double2 y = s_y[buf][rhs][4 * t + kq];
                if (SCALED) {
                    P = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, lx, P, 0, 0, 0);
                    Q = __builtin_amdgcn_mfma_f64_16x16x4f64(y.y, ly, Q, 0, 0, 0);
                    R = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x + y.y, lx + ly, R, 0, 0, 0);
                } else {
                    P = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, lx, P, 0, 0, 0);
                    R = __builtin_amdgcn_mfma_f64_16x16x4f64(y.y, lx, R, 0, 0, 0);
                    P = __builtin_amdgcn_mfma_f64_16x16x4f64(-y.y, ly, P, 0, 0, 0);
                    R = __builtin_amdgcn_mfma_f64_16x16x4f64(y.x, ly, R, 0, 0, 0);
                }
            });
        };

        // this lane: row `row`, columns kq + 4 v
        double cr[4], ci[4];
        uint64_t *in = cols_of(a.in, bi);
        if (SCALED) {  // c = D^-1 b
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint64_t *p = in + (wave + 4 * e) * 2 * TB + lane;
                s_y[0][wave + 4 * e][lane] =
                    make_double2(__longlong_as_double((long long)p[0]), __longlong_as_double((long long)p[TB]));
                if (!UPPER) p[0] = p[TB] = kPsEmpty;
            }
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const double2 d = D[row + (size_t)(4 * t + kq) * TB];
                lcur[t].x = (T)d.x;
                lcur[t].y = (T)d.y;
            }
            __syncthreads();
            product(lcur, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                cr[v] = P[v] - Q[v];
                ci[v] = R[v] - P[v] - Q[v];
            }
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                cr[v] = ci[v] = 0.0;
                if (kq + 4 * v < w) {
                    uint64_t *p = in + (kq + 4 * v) * 2 * TB + row;
                    cr[v] = __longlong_as_double((long long)p[0]);
                    ci[v] = __longlong_as_double((long long)p[TB]);
                    if (!UPPER) p[0] = p[TB] = kPsEmpty;
                }
            }
        }
        auto subtract = [&]() {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                cr[v] -= SCALED ? P[v] - Q[v] : P[v];
                ci[v] -= SCALED ? R[v] - P[v] - Q[v] : R[v];
            }
        };
        // Two blocks per turn, loads without a condition (past the end: the last
        // block once more), so that a product's wait counts leave the next block's
        // loads in flight; an odd block goes first.
        int q = noff & 1;
        if (q) {
            load_block(blk(0), lnext);
            if (!SHORT) load_block(blk(min(1, noff - 1)), lcur);
            __syncthreads();
            product(lnext, 1);
            subtract();
        } else if (!SHORT && noff > 0) {
            load_block(blk(0), lcur);
        }
        for (; !SHORT && q < noff; q += 2) {
            load_block(blk(q + 1), lnext);
            __syncthreads();
            product(lcur, (q + 1) & 1);
            subtract();
            load_block(blk(min(q + 2, noff - 1)), lcur);
            __syncthreads();
            product(lnext, q & 1);
            subtract();
        }
        if (SCALED) {
            uint64_t *o = cols_of(a.pub, bi) + row;
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (kq + 4 * v < w) {
                    put(o + (kq + 4 * v) * 2 * TB, cr[v]);
                    put(o + (kq + 4 * v) * 2 * TB + TB, ci[v]);
                }
            return;
        }
        // into the buffer that no product reads any more
#pragma unroll
        for (int v = 0; v < 4; ++v) s_y[(noff + 1) & 1][kq + 4 * v][row] = make_double2(cr[v], ci[v]);
    }
    if (SCALED) return;

    // Diagonal block: lane = row, wave v has columns v and v + 8.  The
    // substitution is the launch's critical path: unrolled, and without
    // branches.  A step broadcasts row j's value (every lane scales it by the
    // diagonal's reciprocal), and the rows that it reaches take the difference
    // by selection: the others read some entry of the packed block and drop
    // the product, so a step's LDS reads need no mask and are issued ahead.
    // Solving four rows' own triangle in every lane to save broadcasts costs
    // more instructions than the broadcasts: 1103 us per triangle of two
    // matrices with 8 columns at N = 8192 instead of 896.
    __syncthreads();
    auto scaled = [](double2 c, double2 r) { return make_double2(c.x * r.x - c.y * r.y, c.x * r.y + c.y * r.x); };
    auto substitute = [&](auto rw_c) {
        constexpr int RW = decltype(rw_c)::value;
        double2 x[RW];
#pragma unroll
        for (int k = 0; k < RW; ++k) x[k] = s_y[(noff + 1) & 1][wave + 8 * k][lane];
#pragma unroll
        for (int jj = 0; jj < TB; ++jj) {
            const int j = UPPER ? TB - 1 - jj : jj;
            const double2 l = s_d[kPad + (UPPER ? du_idx(lane, j) : dl_idx(lane, j))];
            const double2 ri = UNIT ? make_double2(1.0, 0.0) : s_rd[j];
#pragma unroll
            for (int k = 0; k < RW; ++k) {
                double2 xj = make_double2(bcast(x[k].x, j), bcast(x[k].y, j));
                if (!UNIT) xj = scaled(xj, ri);
                double2 v = x[k];
                cfms(v, l, xj);
                const bool below = UPPER ? lane < j : lane > j;
                x[k].x = below ? v.x : x[k].x;
                x[k].y = below ? v.y : x[k].y;
            }
        }
        if (!UNIT) {  // the rows' own values, as their steps scaled them
#pragma unroll
            for (int k = 0; k < RW; ++k) x[k] = scaled(x[k], s_rd[lane]);
        }
#pragma unroll
        for (int k = 0; k < RW; ++k) {
            const int r = wave + 8 * k;
            if (r >= w) break;
            uint64_t *o = cols_of(a.pub, bi) + r * 2 * TB + lane;
            put(o, x[k].x);
            put(o + TB, x[k].y);
        }
    };
    if (w > 8) substitute(std::integral_constant<int, 2>{});
    else if (wave < w) substitute(std::integral_constant<int, 1>{});
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

// Preconditioner factors: every row block of L and U times the inverse of its
// diagonal block, L' = diag(L_ii)^-1 L and U' = diag(U_ii)^-1 U, so that a solve
// needs no work on the diagonal between one block's values and the next's.
// blockIdx = (column block, row block, slot); row block bi of factor fidx[z],
// column block cb (left of the diagonal: L, right of it: U) is multiplied by
// its inverse on the matrix cores (three real products per complex product,
// lanes as in k_trsv) and written to dst, which may be the factors themselves.
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

// Right-hand sides handled by one residual pass starting at r_off
inline int rhs_chunk(int left) { return left >= 8 ? 8 : left >= 4 ? 4 : left >= 2 ? 2 : 1; }

// Right-hand sides of a pass into its layout: columns r_off ... of each item of B
// (or the columns cols[item * ncols + j], element offsets; -1: zero), rows
// through perm (or as they are), and the solved values' words marked empty.
__global__ void k_rhs_in(const double2 *B, int n, int ldb, int64_t strideB, int r_off, int ncols, const int64_t *cols,
                         const int *perm, int64_t strideQ, const int *bidx, const int *aidx, uint64_t *in,
                         uint64_t *pub)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * ncols) return;
    const int item = blockIdx.y, j = (int)(t / TB % ncols), b = bidx ? bidx[item] : item;
    const int row = (int)(t / ((int64_t)TB * ncols)) * TB + (int)(t % TB);
    const int src = perm ? perm[(size_t)(aidx ? aidx[item] : b) * strideQ + row] : row;
    const int64_t c = cols ? cols[(size_t)item * ncols + j] : (int64_t)b * strideB + (int64_t)(r_off + j) * ldb;
    const size_t o = ((size_t)item * n * ncols + (size_t)(t / TB) * TB) * 2 + t % TB;
    const double2 v = c >= 0 ? B[c + src] : make_double2(0.0, 0.0);
    in[o] = (uint64_t)__double_as_longlong(v.x);
    in[o + TB] = (uint64_t)__double_as_longlong(v.y);
    pub[o] = pub[o + TB] = kPsEmpty;
}

// The solved values back to B, rows through perm (x = P^T w) or as they are.
__global__ void k_rhs_out(const double *x, int n, int ldb, int64_t strideB, int r_off, int ncols, const int64_t *cols,
                          const int *perm, int64_t strideQ, const int *bidx, const int *aidx, double2 *B)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * ncols) return;
    const int item = blockIdx.y, j = (int)(t / TB % ncols), b = bidx ? bidx[item] : item;
    const int row = (int)(t / ((int64_t)TB * ncols)) * TB + (int)(t % TB);
    const int dst = perm ? perm[(size_t)(aidx ? aidx[item] : b) * strideQ + row] : row;
    const int64_t c = cols ? cols[(size_t)item * ncols + j] : (int64_t)b * strideB + (int64_t)(r_off + j) * ldb;
    const size_t o = ((size_t)item * n * ncols + (size_t)(t / TB) * TB) * 2 + t % TB;
    if (c >= 0) B[c + dst] = make_double2(x[o], x[o + TB]);
}

template <typename T, bool TRANS, bool SCALED>
void launch_trsv(const TrsvArgs &a, int items, bool upper, hipStream_t s)
{
    const dim3 grid((unsigned)(items * a.chunks), (unsigned)(a.n / TB)), block(256 + 64 * kPsPoll);
    if (!SCALED && a.n <= 2 * TB) {  // at three blocks a chain's next block is worth loading ahead
        if (upper) hipLaunchKernelGGL((k_trsv<T, true, TRANS, false, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_trsv<T, false, TRANS, false, true>), grid, block, 0, s, a);
        return;
    }
    if (upper) hipLaunchKernelGGL((k_trsv<T, true, TRANS, SCALED, false>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_trsv<T, false, TRANS, SCALED, false>), grid, block, 0, s, a);
}

}  // namespace

int perm_batched(wm_ctx *ctx, int n, const int *ipiv, int64_t strideP, int *perm, int64_t strideQ, int batch,
                 hipStream_t s, const int *d_bidx, void *maps)
{
    // the accepted range of n: as many rows as ints in the LDS (40960).  The kernels
    // below keep no row in LDS; the range is part of the entry points' contract
    if ((size_t)n * sizeof(int) > ctx->max_lds) {
        set_error("permutation: n=%d exceeds %zu rows", n, ctx->max_lds / sizeof(int));
        return WM_ERR_ARG;
    }
    const unsigned nb = (unsigned)((n + 255) / 256);
    if (n <= kPermWhole) {
        hipLaunchKernelGGL(k_perm, dim3(nb, 1, (unsigned)batch), dim3(256), 0, s, ipiv, strideP, n, (n + 63) / 64 * 64,
                           perm, strideQ, d_bidx, 0);
    } else {
        if (!maps) {
            WM_TRY(ctx->ws_solve.ensure((size_t)batch * kPermParts * n * sizeof(int)));
            maps = ctx->ws_solve.ptr;
        }
        const int len = (n + kPermParts * 64 - 1) / (kPermParts * 64) * 64;
        hipLaunchKernelGGL(k_perm, dim3(nb, kPermParts, (unsigned)batch), dim3(256), 0, s, ipiv, strideP, n, len,
                           (int *)maps, (int64_t)n, d_bidx, 1);
        hipLaunchKernelGGL(k_perm_join, dim3(nb, (unsigned)batch), dim3(256), 0, s, (const int *)maps, n, perm,
                           strideQ, d_bidx);
    }
    WM_HIP_TRY(hipGetLastError());
    return WM_OK;
}

namespace {

// Bytes of a solve's right-hand sides and solved values, one pass of them.
size_t solve_bytes(int n, int nrhs, int batch)
{
    return 2 * (size_t)batch * n * std::min(nrhs, kPassCols) * sizeof(double2);
}

// Columns of each matrix in passes of up to kPassCols, in members of up to kPsW
// columns (as even as possible).  trans: solve A^H X = B instead of A X = B.
// ext: the buffer of solve_bytes, supplied by the caller instead of the
// context's (nothing allocated, no profiler events).
int getrs_any(wm_ctx *ctx, int prec, int n, int nrhs, const void *A, int lda, int64_t strideA, const int *perm,
              int64_t strideQ, void *B, int ldb, int64_t strideB, int batch, hipStream_t s, const int *d_bidx,
              bool trans, const int *d_aidx, void *ext = nullptr)
{
    if (n <= 0 || n % TB != 0 || nrhs <= 0 || batch <= 0 || ldb < n) {
        set_error("getrs: bad arguments (n=%d multiple of %d, nrhs=%d, batch=%d)", n, TB, nrhs, batch);
        return WM_ERR_ARG;
    }
    uint64_t *in = (uint64_t *)ext;
    if (!ext) {
        WM_TRY(ctx->ws_solve.ensure(solve_bytes(n, nrhs, batch)));
        in = (uint64_t *)ctx->ws_solve.ptr;
    }
    for (int r0 = 0; r0 < nrhs; r0 += kPassCols) {
        const int nc = std::min(nrhs - r0, kPassCols);
        uint64_t *pub = in + (size_t)batch * n * nc * 2;
        const dim3 vgrid((unsigned)(((int64_t)n * nc + 255) / 256), (unsigned)batch);
        hipLaunchKernelGGL(k_rhs_in, vgrid, dim3(256), 0, s, (const double2 *)B, n, ldb, strideB, r0, nc,
                           (const int64_t *)nullptr, trans ? (const int *)nullptr : perm, strideQ, d_bidx, d_aidx, in,
                           pub);
        TrsvArgs a = {};
        a.A = A; a.lda = lda; a.strideA = strideA; a.n = n; a.ncols = nc; a.err = ctx->d_err;
        a.chunks = (nc + kPsW - 1) / kPsW;
        a.cw = (nc + a.chunks - 1) / a.chunks;
        a.bidx = d_bidx;
        a.aidx = d_aidx;
        const double esz = prec == WM_PREC_F64 ? 16.0 : 8.0;
        const double fl = batch * 4.0 * (double)n * n * nc, by = batch * 0.5 * (double)n * n * esz;
        for (int up = 0; up < 2; ++up) {
            a.in = up ? pub : in;
            a.pub = up ? in : pub;
            if (!ext) prof_begin(ctx, K_TRSV, s);
            if (prec == WM_PREC_F64) {
                if (trans) launch_trsv<double, true, false>(a, batch, up, s);
                else launch_trsv<double, false, false>(a, batch, up, s);
            } else {
                if (trans) launch_trsv<float, true, false>(a, batch, up, s);
                else launch_trsv<float, false, false>(a, batch, up, s);
            }
            if (!ext) prof_end(ctx, K_TRSV, s, fl, by);
        }
        hipLaunchKernelGGL(k_rhs_out, vgrid, dim3(256), 0, s, (const double *)in, n, ldb, strideB, r0, nc,
                           (const int64_t *)nullptr, trans ? perm : (const int *)nullptr, strideQ, d_bidx, d_aidx,
                           (double2 *)B);
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
    WM_TRY(ctx->ws_group.ensure(tab_b + cols_b + 2 * vec_b));
    char *base = (char *)ctx->ws_group.ptr;
    std::vector<char> host(tab_b + cols_b, 0);
    std::memcpy(host.data(), tab.data(), tab.size() * sizeof(int));
    std::memcpy(host.data() + tab_b, cols.data(), cols.size() * sizeof(int64_t));
    WM_TRY(copy_h2d(base, host.data(), host.size(), s));
    const int *d_tab = (const int *)base;
    const int64_t *d_cols = (const int64_t *)(base + tab_b);
    uint64_t *in = (uint64_t *)(base + tab_b + cols_b), *pub = in + vec_b / sizeof(uint64_t);
    const dim3 vgrid((unsigned)(n * kPsW / 256), (unsigned)members);
    hipLaunchKernelGGL(k_rhs_in, vgrid, dim3(256), 0, s, (const double2 *)V, n, n, (int64_t)0, 0, kPsW, d_cols, perm,
                       strideQ, (const int *)nullptr, d_tab, in, pub);
    TrsvArgs a = {};
    a.A = Fs; a.lda = lda; a.strideA = strideF; a.n = n; a.ncols = a.cw = kPsW; a.chunks = 1; a.dinv = Dinv;
    a.aidx = d_tab; a.slot = d_tab + members; a.width = d_tab + 2 * members;
    a.err = ctx->d_err;
    const double fl = 4.0 * (double)n * n * items.size() * nr, by = members * 8.0 * (double)n * n;
    for (int up = 0; up < 2; ++up) {
        a.in = up ? pub : in;
        a.pub = up ? in : pub;
        prof_begin(ctx, K_TRSV, s);
        launch_trsv<double, false, true>(a, members, up, s);
        prof_end(ctx, K_TRSV, s, fl, by);
    }
    hipLaunchKernelGGL(k_rhs_out, vgrid, dim3(256), 0, s, (const double *)in, n, n, (int64_t)0, 0, kPsW, d_cols,
                       (const int *)nullptr, (int64_t)0, (const int *)nullptr, (const int *)nullptr, V);
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
// Allocation-free triangular solves: the permutation and the values' buffers of wm_getrs_batched live in `scratch`, a file-scope device array of
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
    // the documented budget; the values of a pass (solve_bytes) always fit in it:
    // 32 min(nrhs, 32) <= 16 nrhs + 64 nr' bytes per row
    int nr2 = 1;
    while (nr2 * 2 <= std::min(nrhs, 8)) nr2 *= 2;
    const size_t need = perm_b + up((size_t)batch * strideB * sizeof(double2)) + up((size_t)batch * n * nr2 * 64);
    if (need > kNoAllocBytes) {
        set_error("wm_getrs_batched_noalloc: n=%d, nrhs=%d, batch=%d need %zu bytes of scratch, the maximum is %zu "
                  "(use wm_getrs_batched)", n, nrhs, batch, need, kNoAllocBytes);
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
    // the parts' maps (32 bytes per row) lie where the values go afterwards (32 per row and column)
    WM_TRY(perm_batched(ctx, n, ipiv, strideP, perm, n, batch, s, nullptr, base + perm_b));
    WM_TRY(getrs_any(ctx, prec, n, nrhs, A, lda, strideA, perm, n, B, ldb, strideB, batch, s, nullptr, false, nullptr,
                     base + perm_b));
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
