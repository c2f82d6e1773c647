// Batched dense complex LU with partial pivoting for gfx950.
//
// Replaces the reference's LAPACKE_zgetrf ("wersja referencyjna/Wire_MoM.cu":372,
// MKL) and cublasZgetrfBatched ("wersja gpu/Wire_MoM.cu":468).  Same contract
// as LAPACK zgetrf: column-major, pivot = first row with the largest
// |re|+|im| in the column (izamax), 1-based ipiv, info = first exactly-zero
// pivot, rows interchanged across the whole matrix.
//
// Blocked right-looking algorithm with panel width NB = 64, in outer blocks
// of kSub panels.  Per panel k:
//   1. k_panel      : GEPP of the n-k x NB panel.  A cluster of P workgroups
//                     per matrix holds the panel in registers (a row split
//                     over four threads, two for complex64); per column the
//                     workgroups exchange their pivot candidates through
//                     tagged packets, all reduce them to the same pivot,
//                     relabel and apply the rank-1 update locally.  It
//                     also emits the composite row permutation of the panel.
//   2. k_swap_trsm  : applies that permutation to the columns outside the
//                     panel and computes U12 = L11^{-1} A12 for the outer
//                     block's remaining columns (forward substitution, L11
//                     from LDS).
//   3. k_gemm_*     : A -= L U on the matrix cores, with three real products
//                     per complex product: complex128 with
//                     v_mfma_f64_16x16x4f64, complex64 with
//                     v_mfma_f32_32x32x2f32, or with split-bf16 operands and
//                     v_mfma_f32_32x32x16_bf16.  Inside an outer block a
//                     short product brings the later panels' rows up to
//                     date; one product with K = 64 kSub updates the
//                     trailing matrix per outer block.  The MFMA is issued on
//                     the transposed problem (C^T = U^T L^T) so each lane's
//                     accumulator column is a run of consecutive rows of C:
//                     the C read-modify-write is coalesced in column-major
//                     storage.
#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <vector>

#include "wm_cplx.h"
#include "wm_internal.h"

namespace wm {

namespace {

constexpr int NB = 64;
// Panels per outer block of the factorization (tunable per context).  Deeper
// blocks give the trailing update a longer K (better MFMA use) at the cost of
// more narrow updates inside the block.  At N = 8192 8 panels beat 4 by 1.4-6.5 %
// while the narrow updates were slow; now 4 are ahead there (2 x 8192 complex128
// 69.7 against 72.3 ms, 10 x 8192 split-BF16x3 113.7 against 115.2; 2 x 14336 265.1
// against 265.9).  The defaults are what wm_get_getrf_block reports and stay;
// wm_tune_getrf finds the faster depth.
constexpr int kSubDefault = 4, kSubLarge = 8, kSubLargeN = 8192;
// Parts per panel row (waves sharing a row).  Narrow parts shorten what each
// wave does per column (16 or 32 columns of updates, the transposition of a
// candidate row); complex128 panels measured 208 us with two parts (3 -> 2
// workgroups per CU) and 165 us with four, complex64 ones 280 us with one and
// 196 us with two (64 columns, N = 512 .. 4096).
// Half as many parts, and rows of twice as many columns per thread, take a matrix
// whose clusters do not fit on the device otherwise (rows above 64, complex64 128,
// per resident workgroup: 12288 complex128 rows where four contexts share the
// device), in a kernel of its own (k_panel_tall).
constexpr int kTprF64 = 4, kTprF32 = 2;

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// Panel exchange buffers.  The workgroups of one panel cluster talk through
// 8-byte packets {32-bit payload, 32-bit tag}; the tag names the column (a
// per-launch base plus the column index, never reused while the buffer lives),
// so a reader polls each packet until its tag matches and no fence or counter
// is needed: 8-byte loads and stores are single-copy atomic, and agent-scope
// relaxed atomics go to the device coherence point without flushing caches.
// Packets alternate between two buffers by column parity: a workgroup
// publishes column j+2 only after reading all packets of column j+1, which
// every workgroup published after its reads of column j.
//
// Per launch member and parity:
//   slot [slots][SLS]: |candidate| as two 32-bit halves of a double, its position, unused
//   cand [slots][NWS]: each candidate's row (NW 32-bit words, per chunk the low
//                     or real halves of its 32 values, then the high or
//                     imaginary ones) and the reciprocal of its pivot (4 words)
// followed by kPermSlots panel permutations (one per panel of an outer block):
// cnt, rows[2NB], src[2NB].
constexpr int kPermSlots = 16;  // panels per outer block at most
template <typename V>
struct XLayout {
    static constexpr int NW = NB * (int)sizeof(V) / 4;  // 32-bit words per panel row
    static constexpr int NWS = NW + 16;  // stride of the candidate rows (whole 128-byte lines)
    static constexpr int SLS = 4;        // stride of the slots: dense, a poll reads few lines
    size_t par_bytes, perm_off, mat_bytes;
    int slots;  // candidates per column: one per wave of 64 rows (k_panel_tall: one per workgroup)
    __host__ __device__ XLayout(int slots_) : slots(slots_)
    {
        par_bytes = (size_t)slots * (SLS + NWS) * sizeof(uint64_t);
        par_bytes = (par_bytes + 255) & ~(size_t)255;
        perm_off = 2 * par_bytes;
        mat_bytes = perm_off + kPermSlots * (1 + 4 * NB) * sizeof(int);
        mat_bytes = (mat_bytes + 255) & ~(size_t)255;
    }
    __device__ uint64_t *slot(char *m, int par) const { return (uint64_t *)(m + par * par_bytes); }
    __device__ uint64_t *cand(char *m, int par) const { return slot(m, par) + (size_t)slots * SLS; }
    __device__ int *perm(char *m, int slot) const { return (int *)(m + perm_off) + slot * (1 + 4 * NB); }
};

// Columns of the panel updated together, and workgroups per CU that the
// register allocation allows for (4 per CU, 128 registers, spill: 205 against
// 159 us per complex128 panel).
constexpr int kPanelGroup = 4, kPanelOcc = 3;

template <typename T>
struct PanelArgs {
    typename CT<T>::V *A;
    int lda;
    int64_t strideA;
    int n, k, P, slots;
    int pslot;  // where the panel's permutation goes
    int *ipiv;
    int64_t strideP;
    int *info;
    int *err;
    char *xbuf;
    const int *bidx;  // launch member -> matrix index (null: identity)
    const uint32_t *tagp;  // device tag base of the current factorization (bumped per launch chunk)
    uint32_t toff;         // packet tags of this launch are *tagp + toff + 1 .. *tagp + toff + NB
    const int *nmem;       // per matrix index: its own size (rows/columns beyond are the identity), or null
};

// Argmax combine: larger value wins, equal values go to the lower row.
__device__ inline bool better(double v2, int r2, double v1, int r1) { return v2 > v1 || (v2 == v1 && r2 < r1); }

// Cross-lane moves within rows of 16 lanes (DPP: quad permutations and row
// rotations, every source lane valid).
template <int CTRL>
__device__ inline int dpp_i32(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
__device__ inline double readlane_f64(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Reductions over the wave (quad_perm [1,0,3,2], [2,3,0,1], row_ror 4, row_ror 8,
// then the four rows' results); every lane gets the result.
__device__ inline int wave_min_i32(int v)
{
    v = min(v, dpp_i32<0xB1>(v));
    v = min(v, dpp_i32<0x4E>(v));
    v = min(v, dpp_i32<0x124>(v));
    v = min(v, dpp_i32<0x128>(v));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

__device__ inline int wave_max_i32(int v)
{
    v = max(v, dpp_i32<0xB1>(v));
    v = max(v, dpp_i32<0x4E>(v));
    v = max(v, dpp_i32<0x124>(v));
    v = max(v, dpp_i32<0x128>(v));
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

constexpr int kNoRow = 0x7fffffff;

// Lane with the largest v >= 0 among those with cand (the lowest position on
// ties; v of a candidate is not NaN), or -1.  The high words of non-negative
// doubles order as integers, so one 32-bit reduction decides unless two
// candidates agree in them (or there is none).
__device__ inline int wave_best(double v, int pos, bool cand)
{
    const long long bits = __double_as_longlong(v);
    const int hi = cand ? (int)(bits >> 32) : -1;
    const int m = wave_max_i32(hi);
    unsigned long long t = __ballot(hi == m);
    if (t & (t - 1)) {
        // the low words as signed integers in the order of unsigned ones; every
        // lane takes part in the reductions
        bool in = cand && hi == m;
        const int lo = in ? (int)((unsigned)bits ^ 0x80000000u) : (int)0x80000000;
        const int lm = wave_max_i32(lo);
        in = in && lo == lm;
        const int first = wave_min_i32(in ? pos : kNoRow);
        in = in && pos == first;
        t = __ballot(in);
    }
    return t ? (int)__builtin_ctzll(t) : -1;
}

__device__ inline double readlane_t(double v, int l) { return readlane_f64(v, l); }
__device__ inline float readlane_t(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// (re, im) - (lr, li) * (ur, ui): the complex product is rounded before it is
// subtracted.  Fused into the subtraction it would save a third of the
// operations, but wire matrices eliminate by exact cancellations (their
// charge terms): with l = x / p, a rounded l * p gives x back where the fused
// form keeps l's rounding error, and Zin of a 1024-unknown grid at 1 MHz came
// out 100 times less accurate (1.9e-10 instead of 2e-12).
template <typename T>
__device__ inline T sub_mul_re(T re, T lr, T li, T ur, T ui)
{
#pragma clang fp contract(off)
    const T p = li * ui;
    return re - fma_t(lr, ur, -p);
}
template <typename T>
__device__ inline T sub_mul_im(T im, T lr, T li, T ur, T ui)
{
#pragma clang fp contract(off)
    const T p = lr * ui;
    return im - fma_t(li, ur, p);
}
// (ar, ai) * (br, bi), rounded alike
__device__ inline double2 mul_c(double ar, double ai, double br, double bi)
{
#pragma clang fp contract(off)
    const double p = ai * bi, q = ar * bi;
    return make_double2(fma_t(ar, br, -p), fma_t(ai, br, q));
}

// Composite permutation of a panel's interchanges, for the other columns, by the
// first wave of workgroup 0: after applying them in order, row rows[t] holds the
// old content of src[t].  Slots t < NB are rows k + t; the rows from below the
// panel that take part get slots NB, NB+1, ... in order of first use.  The wave
// keeps pivot t, slot t and slot NB + t in lane t (NB is the wave width), so each
// interchange is a ballot and three lane reads.
__device__ inline void panel_perm(int k, int lane, const int *s_piv, int *pm)
{
    static_assert(NB == 64, "one slot pair per lane");
    const int rlo = k + lane;
    int slo = k + lane, rhi = -1, shi = -1;
    const int pv = s_piv[lane];  // pivot row of column `lane`
    int cnt = NB;
    for (int jx = 0; jx < NB; ++jx) {
        const int pp = __builtin_amdgcn_readlane(pv, jx);
        if (pp == k + jx) continue;
        int tp;
        if (pp < k + NB) {
            tp = pp - k;
        } else {
            const unsigned long long hit = __ballot(NB + lane < cnt && rhi == pp);
            if (hit) {
                tp = NB + (int)__builtin_ctzll(hit);
            } else {
                tp = cnt++;
                if (lane == tp - NB) { rhi = pp; shi = pp; }
            }
        }
        const int sj = __builtin_amdgcn_readlane(slo, jx);
        const int st = tp < NB ? __builtin_amdgcn_readlane(slo, tp) : __builtin_amdgcn_readlane(shi, tp - NB);
        if (lane == jx) slo = st;
        if (tp < NB) {
            if (lane == tp) slo = sj;
        } else if (lane == tp - NB) {
            shi = sj;
        }
    }
    int *rows = pm + 1, *src = pm + 1 + 2 * NB;
    rows[lane] = rlo;
    src[lane] = slo;
    if (NB + lane < cnt) {
        rows[NB + lane] = rhi;
        src[NB + lane] = shi;
    }
    if (lane == 0) pm[0] = cnt;
}

// GEPP of the (n-k) x NB panel at column k for one matrix per blockIdx.y.
// Workgroup w holds rows k + w*RW .. k + (w+1)*RW - 1 in registers.  A row is
// split into TPR parts of W = NB/TPR columns held by different waves ("chunk"
// c = wave / NWC), so that within a wave the column index is uniform: only
// the waves owning column j take part in its argmax (a DPP reduction), and
// each thread carries its row's value in the next pivot column (nxr, nxi),
// taken from the update that produces it, so registers are only indexed
// statically.
//
// Interchanges move labels, not data: each thread keeps its row and carries
// the row's current position lr (initially the row itself).  Exchanging rows
// k+j and gr swaps the two labels; the row labelled k+j is the pivot row and
// is final from then on, the rows labelled above k+j take the rank-1 update.
// The arithmetic and the pivots are those of the interchanging algorithm
// (ties go to the lowest position, as izamax), and each row is stored at its
// final position at the end.
//
// A column costs a chain of latencies, not work (the panel's flops would take
// a few microseconds on the CUs it occupies), so the chain is kept short:
//  * each wave publishes its own candidate's slot as soon as its argmax is
//    known, and its row right after: the candidate row is transposed through
//    LDS, so that one lane per value brings it up to date (by the last column)
//    and publishes it, before the wave updates all its rows;
//  * that update (of the columns right of j by column j-1) and the reciprocal
//    of the candidate's pivot run while the slots travel.  The update walks
//    groups of G columns without branches, so a group's pivot-row reads from
//    LDS are in flight together (a branch per column made each read's latency
//    serial: half the time of a column);
//  * after the pivot is known only its column's multipliers and the next
//    column's values are computed before the next argmax;
//  * the row of slot 0 is polled along with the slots, so a pivot near the
//    diagonal (995 of 1000 columns of the wire matrices) costs one round trip;
//  * a cluster of one workgroup exchanges nothing.
// Measured per 64-column complex128 panel, pivots near the diagonal: 341 -> 144
// us (one matrix of N = 512), 348 -> 158 us (two, N = 8192), 418 -> 204 us (16,
// N = 8192, three workgroups per CU); random pivots 352 -> 165, 356 -> 180, 430
// -> 225 us; complex64 panels (12 of N = 8192) 433 -> 207 us.  What is left of
// a column's 2.3 us: the argmax and the candidate row (0.8 us), the packets'
// way to memory and back (0.9 us; the same inside one XCD), the pivot row to
// all waves and the next column (0.3 us).
template <typename T, int TPR>
__global__ __launch_bounds__(256, kPanelOcc) void k_panel(PanelArgs<T> a)
{
    using V = typename CT<T>::V;
    constexpr int W = NB / TPR;     // columns per thread
    constexpr int NWC = 4 / TPR;    // waves per chunk: candidates per workgroup
    constexpr int RW = 64 * NWC;    // rows per workgroup
    constexpr int NW = XLayout<V>::NW, NWS = XLayout<V>::NWS, SLS = XLayout<V>::SLS;
    constexpr int G = kPanelGroup;  // columns updated together
    constexpr int NE = NW / TPR / 2;  // values of a chunk's part of a row: one lane each (complex128: re and im apart)
    static_assert((NE == 32 || NE == 64) && TPR > 1 && RW >= NB && W % 8 == 0 && W % G == 0, "panel layout");
    const int bl = blockIdx.y, w = blockIdx.x;          // bl: member of this launch
    const int b = a.bidx ? a.bidx[bl] : bl;              // b: matrix index
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = wave / NWC, rb = wave % NWC;           // chunk (columns c*W ..), row block
    const int k = a.k, base = k + w * RW;
    const int row = base + rb * 64 + lane;
    const bool valid = row < a.n;
    V *Ab = a.A + (size_t)b * a.strideA;
    const XLayout<V> X(a.slots);
    char *xm = a.xbuf + (size_t)bl * X.mat_bytes;
    if (a.nmem && k >= a.nmem[b]) {
        // the member's own matrix ends above this panel: an identity panel, no
        // interchanges (pivots k+1 .. k+NB) and an empty permutation
        if (w == 0 && tid < NB) a.ipiv[(size_t)b * a.strideP + k + tid] = k + tid + 1;
        if (w == 0 && tid == 0) X.perm(xm, a.pslot)[0] = 0;
        return;
    }

    T re[W], im[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        V x = V{0, 0};
        if (valid) x = Ab[row + (size_t)(k + c * W + i) * a.lda];
        re[i] = x.x;
        im[i] = x.y;
    }

    // s_u, s_nx and the pivot's data alternate with the column parity: a wave
    // may still use column j-1's pivot row while wave 0 writes column j's
    __shared__ double s_wv[NWC];
    __shared__ int s_wr[NWC], s_wl[NWC];    // each row block's candidate: value, position, lane (-1: none)
    __shared__ T s_cand[NWC][2][NB];        // its row, real and imaginary parts
    __shared__ V s_u[2][NB];                // pivot row
    __shared__ V s_nx[2][RW];               // values in the pivot column, for the other chunks
    __shared__ double s_gv[2];
    __shared__ int s_gr[2];
    __shared__ double2 s_rinv[2];           // reciprocal of the pivot
    __shared__ int s_piv[NB];               // pivot row of each column (workgroup 0)

    const uint32_t tag0 = *a.tagp + a.toff;
    const bool solo = a.P == 1;
    const int nslots = a.P * NWC;
    int lr = row;  // current position of this thread's row
    // this row's value in the column of the next step (column 0 is in chunk 0)
    T nxr = re[0], nxi = im[0];
    T lre = 0, lim = 0;  // this row's multiplier of the last column
    bool act = false;    // this row takes the last column's update
    int zero = -1;       // first column with a zero pivot
    for (int j = 0; j < NB; ++j) {
        const int par = j & 1;
        const int pr = k + j;
        const int cj = j / W;
        const uint32_t tag = tag0 + (uint32_t)j + 1u;
        uint64_t *slot = X.slot(xm, par);
        uint64_t *cand = X.cand(xm, par);

        // 1. best row of each wave of the chunk holding column j: largest
        //    |re|+|im| among positions >= k+j, the lowest position on ties
        //    (NaN is never a candidate); its slot is published at once
        if (c == cj) {
            const double v = fabs((double)nxr) + fabs((double)nxi);
            const int l = wave_best(v, lr, valid && lr >= pr && v == v);
            const int ll = max(l, 0);
            const double wv = l < 0 ? -1.0 : readlane_f64(v, ll);
            const int wr = l < 0 ? kNoRow : __builtin_amdgcn_readlane(lr, ll);
            if (!solo && lane < 3) {  // one store of three packets
                const uint64_t bits = (uint64_t)__double_as_longlong(wv);
                const uint32_t word = lane == 0 ? (uint32_t)bits : lane == 1 ? (uint32_t)(bits >> 32) : (uint32_t)wr;
                put_pkt(slot + (w * NWC + rb) * SLS + lane, tag, word);
            }
            if (lane == 0) {
                s_wl[rb] = l;
                if (solo) {
                    s_wv[rb] = wv;
                    s_wr[rb] = wr;
                }
            }
            s_nx[par][rb * 64 + lane] = V{nxr, nxi};
        }
        __syncthreads();
        const int wl = __builtin_amdgcn_readfirstlane(s_wl[rb]);

        // 2. the candidate's row from column j on, brought up to date, and the
        //    reciprocal of its pivot; in a cluster of one workgroup the best
        //    row block's is the pivot row
        bool owner = true;
        if (solo) {
            double bv = s_wv[0];
            int br = s_wr[0], bq = 0;
#pragma unroll
            for (int q = 1; q < NWC; ++q)
                if (better(s_wv[q], s_wr[q], bv, br)) { bv = s_wv[q]; br = s_wr[q]; bq = q; }
            owner = rb == __builtin_amdgcn_readfirstlane(bq);
            if (tid == 0) {
                const bool ok = br >= pr && br < a.n;  // else: a zero pivot in place
                s_gv[par] = ok ? bv : 0.0;
                s_gr[par] = ok ? br : pr;
            }
        }
        // the pivot's reciprocal: by a wave whose columns are finished, where
        // there is one
        if (wl >= 0 && owner && c == (cj > 0 ? cj - 1 : 0) && lane == 0) {
            const V p = s_nx[par][rb * 64 + wl];
            const double2 rp = p.x != 0 || p.y != 0 ? crecip((double)p.x, (double)p.y) : make_double2(0.0, 0.0);
            if (solo) {
                s_rinv[par] = rp;
            } else {
                uint64_t *pq = cand + (w * NWC + rb) * NWS + NW;
                const uint64_t xb = (uint64_t)__double_as_longlong(rp.x), yb = (uint64_t)__double_as_longlong(rp.y);
                put_pkt(pq, tag, (uint32_t)xb);
                put_pkt(pq + 1, tag, (uint32_t)(xb >> 32));
                put_pkt(pq + 2, tag, (uint32_t)yb);
                put_pkt(pq + 3, tag, (uint32_t)(yb >> 32));
            }
        }
        if (wl >= 0 && owner && c >= cj) {
            T *dre = s_cand[rb][0] + c * W, *dim = s_cand[rb][1] + c * W;
            const bool upd = j > 0 && (sizeof(T) == 4 || __builtin_amdgcn_readlane((int)act, wl));
            const T wlr = readlane_t(lre, wl), wli = readlane_t(lim, wl);
            if (lane == wl) {
#pragma unroll
                for (int g = 0; g < W; g += 8)
                    if (c * W + g + 7 >= j) {
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            dre[g + q] = re[g + q];
                            dim[g + q] = im[g + q];
                        }
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            uint64_t *pc = cand + (w * NWC + rb) * NWS + 2 * c * NE + lane;
            if constexpr (sizeof(T) == 8) {  // two lanes per column: real and imaginary part
                const bool imag = lane & 1;
                const int i = (lane % NE) / 2, col = c * W + i;
                double x = imag ? dim[i] : dre[i];
                const V u = s_u[par ^ 1][col];
                if (upd) {
                    // sub_mul_re or sub_mul_im
                    x = sub_mul_im(x, imag ? wlr : -wli, imag ? wli : wlr, u.x, u.y);
                }
                if (lane < NE && col >= j) {
                    if (solo) {
                        ((double *)s_u[par])[2 * col + imag] = x;
                    } else {
                        const uint64_t xb = (uint64_t)__double_as_longlong(x);
                        put_pkt(pc, tag, (uint32_t)xb);
                        put_pkt(pc + NE, tag, (uint32_t)(xb >> 32));
                    }
                }
            } else {  // one lane per column
                const int i = lane % NE, col = c * W + i;
                V x = V{dre[i], dim[i]};
                const V u = s_u[par ^ 1][col];
                if (upd) {
                    x = V{sub_mul_re(x.x, wlr, wli, u.x, u.y), sub_mul_im(x.y, wlr, wli, u.x, u.y)};
                }
                if (lane < NE && col >= j) {
                    if (solo) {
                        s_u[par][col] = x;
                    } else {
                        put_pkt(pc, tag, (uint32_t)__float_as_int(x.x));
                        put_pkt(pc + NE, tag, (uint32_t)__float_as_int(x.y));
                    }
                }
            }
        }

        // 3. column j-1's multipliers and its update of the columns from j on.
        //    complex64 factors: rows that take no update have a zero
        //    multiplier, so the update needs no per-row branch (a non-finite
        //    pivot row then spreads to finished rows, and the refinement of
        //    such factors fails over to FP64 factors); complex128 factors keep
        //    LAPACK's untouched finished rows
        if (j > 0 && (sizeof(T) == 4 || act)) {
            const V *su = s_u[par ^ 1] + c * W;
            const int jc = j - 1 - c * W;
            auto upd = [&](int i, const V &u) {
                re[i] = sub_mul_re(re[i], lre, lim, u.x, u.y);
                im[i] = sub_mul_im(im[i], lre, lim, u.x, u.y);
            };
#pragma unroll
            for (int g = 0; g < W; g += G) {
                if (g > jc) {
                    V u[G];
#pragma unroll
                    for (int q = 0; q < G; ++q) u[q] = su[g + q];
#pragma unroll
                    for (int q = 0; q < G; ++q) upd(g + q, u[q]);
                } else if (g + G > jc) {
#pragma unroll
                    for (int q = 0; q < G; ++q) {
                        if (g + q > jc) upd(g + q, su[g + q]);
                        if (g + q == jc && act) {
                            re[g + q] = lre;
                            im[g + q] = lim;
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the next column's values before column j's update
        T xr = 0, xi = 0;
        {
            const int jn = j + 1 - c * W;
#pragma unroll
            for (int g = 0; g < W; g += 8)
                if (jn >= g && jn < g + 8) {
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        if (g + q == jn) {
                            xr = re[g + q];
                            xi = im[g + q];
                        }
                }
        }

        // 4. wave 0 reduces all candidates to the same pivot (first max), then
        //    fetches the pivot row and reciprocal of the winner; one barrier
        //    hands everything to the others
        if (!solo && wave == 0) {
            // The row of slot 0 (the panel's top 64 rows) is polled along with the
            // slots: it is the pivot row in 995 of 1000 columns of the wire
            // matrices, whose pivots stay near the diagonal.
            constexpr int PL = NW / 64;  // pivot-row words per lane, loaded together
            uint64_t wu[PL], wi;
            // the value whose word this lane takes, and which of its two words
            auto val = [&](int e) { return (64 * e + lane) / (2 * NE) * NE + lane % NE; };
            auto half = [&](int e) { return (64 * e + lane) / NE % 2; };
            auto load_row = [&](int sl) {
                const uint64_t *pu = cand + sl * NWS;
#pragma unroll
                for (int e = 0; e < PL; ++e) wu[e] = ld_pkt(pu + lane + 64 * e);
                wi = ld_pkt(pu + NW + (lane & 3));
            };
            auto row_ready = [&]() {
                bool got = (uint32_t)(wi >> 32) == tag;
#pragma unroll
                for (int e = 0; e < PL; ++e)  // columns left of j are not published
                    got = got && ((uint32_t)(wu[e] >> 32) == tag || (sizeof(T) == 8 ? val(e) / 2 : val(e)) < j);
                return __all(got) != 0;
            };
            double gv = -1.0;
            int gr = kNoRow, gs = 0;
            for (int s0 = 0; s0 < nslots; s0 += 128) {  // two slots per lane at a time
                uint64_t w0[2], w1[2], w2[2];
                long it = 0;
                for (;;) {
                    bool got = true;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int s = s0 + 64 * h + lane;
                        if (s < nslots) {
                            const uint64_t *ps = slot + s * SLS;
                            w0[h] = ld_pkt(ps);
                            w1[h] = ld_pkt(ps + 1);
                            w2[h] = ld_pkt(ps + 2);
                        }
                    }
                    load_row(0);
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        if (s0 + 64 * h + lane < nslots)
                            got = got && (uint32_t)(w0[h] >> 32) == tag && (uint32_t)(w1[h] >> 32) == tag &&
                                  (uint32_t)(w2[h] >> 32) == tag;
                    if (__all(got)) break;
                    if (spin_give_up(it, a.err)) break;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int s = s0 + 64 * h + lane;
                    if (s < nslots) {
                        const double v2 = __longlong_as_double(
                            (long long)(((w1[h] & 0xffffffffull) << 32) | (w0[h] & 0xffffffffull)));
                        const int r2 = (int)(uint32_t)w2[h];
                        if (better(v2, r2, gv, gr)) { gv = v2; gr = r2; gs = s; }
                    }
                }
            }
            const int l = wave_best(gv, gr, gr != kNoRow);
            const int r = l >= 0 ? __builtin_amdgcn_readlane(gr, l) : kNoRow;
            // no usable candidate (non-finite column): a zero pivot in place
            const bool ok = r >= pr && r < a.n;
            double2 rinv = make_double2(0.0, 0.0);
            double m = 0.0;
            if (ok) {
                m = readlane_f64(gv, l);
                const int ws = __builtin_amdgcn_readlane(gs, l);
                long it = 0;
                if (ws != 0) load_row(ws);
                while (!row_ready()) {
                    if (spin_give_up(it, a.err)) break;
                    load_row(ws);
                }
#pragma unroll
                for (int e = 0; e < PL; ++e) ((uint32_t *)s_u[par])[2 * val(e) + half(e)] = (uint32_t)wu[e];
                const uint32_t ri = (uint32_t)wi;
                auto word = [&](int q) { return (unsigned long long)(unsigned)__builtin_amdgcn_readlane(ri, q); };
                rinv.x = __longlong_as_double((long long)((word(1) << 32) | word(0)));
                rinv.y = __longlong_as_double((long long)((word(3) << 32) | word(2)));
            }
            if (lane == 0) {
                s_gv[par] = m;
                s_gr[par] = ok ? r : pr;
                s_rinv[par] = rinv;
            }
        }
        __syncthreads();
        const double gv = s_gv[par];
        const int gr = s_gr[par];
        const double2 rinv = s_rinv[par];
        const V un = s_u[par][j + 1 < NB ? j + 1 : j];
        if (c != cj) {
            const V x = s_nx[par][rb * 64 + lane];
            nxr = x.x;
            nxi = x.y;
        }

        // 5. interchange positions k+j and gr, the multipliers of column j,
        //    and the next column's values for the next argmax
        if (tid == 0) s_piv[j] = gr;
        if (gv == 0.0 && zero < 0) zero = pr;
        if (lr == gr) lr = pr;
        else if (lr == pr) lr = gr;
        act = gv != 0.0 && valid && lr > pr;
        lre = lim = 0;
        if (act) {
            const double2 l = mul_c((double)nxr, (double)nxi, rinv.x, rinv.y);
            lre = (T)l.x;
            lim = (T)l.y;
        }
        nxr = xr;
        nxi = xi;
        if (sizeof(T) == 4 || act) {
            nxr = sub_mul_re(xr, lre, lim, un.x, un.y);
            nxi = sub_mul_im(xi, lre, lim, un.x, un.y);
        }
    }
    if (c == TPR - 1 && act) {  // the last column's multipliers
        re[W - 1] = lre;
        im[W - 1] = lim;
    }

    // each row to its final position
#pragma unroll
    for (int i = 0; i < W; ++i)
        if (valid) Ab[lr + (size_t)(k + c * W + i) * a.lda] = V{re[i], im[i]};

    __syncthreads();  // s_piv complete
    if (w == 0 && tid < NB) a.ipiv[(size_t)b * a.strideP + k + tid] = s_piv[tid] + 1;
    if (w == 0 && tid == 0 && zero >= 0 && a.info[b] == 0) a.info[b] = zero + 1;
    if (w == 0 && wave == 0) panel_perm(k, lane, s_piv, X.perm(xm, a.pslot));
}

// The panel of a matrix too tall for k_panel's clusters: twice the rows per
// workgroup (complex128 128 in two parts, complex64 256 in whole rows), the same
// pivots, arithmetic and order, so the same bits.  A thread's 128 registers of
// columns leave 40 at three workgroups per CU, and fewer workgroups would refuse
// matrices that fit now; so nothing is carried from a column to the next but the
// next pivot column's values: one candidate per workgroup, published after a second
// barrier, and the update whole before the next argmax.  k_panel's deferred update
// with this many columns spills 205 (complex128) and 343 registers, which is slow,
// and lane reads among reloads are not safe (a register reloaded for some lanes
// only does not hold the others' values): the build refuses it.  Per 64 columns of
// one matrix of N = 4096 with random pivots 348 us in complex128 (the spilling form
// 497, k_panel 171) and 433 us in complex64 (697, 205).
template <typename T, int TPR>
__global__ __launch_bounds__(256, kPanelOcc) void k_panel_tall(PanelArgs<T> a)
{
    using V = typename CT<T>::V;
    constexpr int W = NB / TPR;     // columns per thread
    constexpr int NWC = 4 / TPR;    // waves per chunk
    constexpr int RW = 64 * NWC;    // rows per workgroup
    constexpr int NW = XLayout<V>::NW, NWS = XLayout<V>::NWS, SLS = XLayout<V>::SLS;
    static_assert(NW <= 256 && NW % 64 == 0 && RW >= NB, "panel layout");
    const int bl = blockIdx.y, w = blockIdx.x;          // bl: member of this launch
    const int b = a.bidx ? a.bidx[bl] : bl;              // b: matrix index
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = wave / NWC, rb = wave % NWC;           // chunk (columns c*W ..), row block
    const int k = a.k, base = k + w * RW;
    const int row = base + rb * 64 + lane;
    const bool valid = row < a.n;
    V *Ab = a.A + (size_t)b * a.strideA;
    const XLayout<V> X(a.slots);
    char *xm = a.xbuf + (size_t)bl * X.mat_bytes;
    if (a.nmem && k >= a.nmem[b]) {  // as in k_panel
        if (w == 0 && tid < NB) a.ipiv[(size_t)b * a.strideP + k + tid] = k + tid + 1;
        if (w == 0 && tid == 0) X.perm(xm, a.pslot)[0] = 0;
        return;
    }

    T re[W], im[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        V x = V{0, 0};
        if (valid) x = Ab[row + (size_t)(k + c * W + i) * a.lda];
        re[i] = x.x;
        im[i] = x.y;
    }

    __shared__ double s_wv[NWC];
    __shared__ int s_wr[NWC];
    __shared__ V s_cand[NB];  // this workgroup's best row
    __shared__ V s_u[NB];     // pivot row
    __shared__ V s_l[TPR > 1 ? RW : 1];  // multipliers for the other chunks
    __shared__ double s_gv;
    __shared__ int s_gr;
    __shared__ double2 s_rinv;  // reciprocal of the pivot
    __shared__ int s_piv[NB];   // pivot row of each column (workgroup 0)
    __shared__ int s_zero;      // first column with a zero pivot
    if (tid == 0) s_zero = -1;

    const uint32_t tag0 = *a.tagp + a.toff;
    int lr = row;  // current position of this thread's row
    // this row's value in the column of the next step (column 0 is in chunk 0)
    T nxr = re[0], nxi = im[0];
    for (int j = 0; j < NB; ++j) {
        const int par = j & 1;
        const int pr = k + j;
        const int cj = j / W;
        const uint32_t tag = tag0 + (uint32_t)j + 1u;

        // 1. best row of each wave of the chunk holding column j
        if (c == cj) {
            const double v = fabs((double)nxr) + fabs((double)nxi);
            const int l = wave_best(v, lr, valid && lr >= pr && v == v);
            const int ll = max(l, 0);
            const double wv = l < 0 ? -1.0 : readlane_f64(v, ll);
            const int wr = l < 0 ? kNoRow : __builtin_amdgcn_readlane(lr, ll);
            if (lane == 0) {
                s_wv[rb] = wv;
                s_wr[rb] = wr;
            }
        }
        __syncthreads();

        // 2. this workgroup's candidate: its slot is published at once, so the
        //    other workgroups' reductions start while the row is staged in LDS
        double wv = s_wv[0];
        int wr = s_wr[0];
#pragma unroll
        for (int q = 1; q < NWC; ++q)
            if (better(s_wv[q], s_wr[q], wv, wr)) { wv = s_wv[q]; wr = s_wr[q]; }
        uint64_t *slot = X.slot(xm, par);
        uint64_t *cand = X.cand(xm, par);
        if (tid < 3) {
            const uint64_t bits = (uint64_t)__double_as_longlong(wv);
            const uint32_t word = tid == 0 ? (uint32_t)bits : tid == 1 ? (uint32_t)(bits >> 32) : (uint32_t)wr;
            put_pkt(slot + (size_t)w * SLS + tid, tag, word);
        }
        if (wr != kNoRow && lr == wr) {
#pragma unroll
            for (int i = 0; i < W; ++i) s_cand[c * W + i] = V{re[i], im[i]};
        }
        __syncthreads();

        // 3. publish the candidate row (its words in the order of memory)
        if (tid < NW) put_pkt(cand + (size_t)w * NWS + tid, tag, ((const uint32_t *)s_cand)[tid]);

        // 4. wave 0 reduces all candidates to the same pivot (first max), then
        //    fetches the pivot row from the workgroup holding it and takes the
        //    pivot's reciprocal, so one barrier hands everything to the others
        if (wave == 0) {
            double gv = -1.0;
            int gr = kNoRow, gs = 0;
            for (int s = lane; s < a.P; s += 64) {
                const uint64_t *ps = slot + (size_t)s * SLS;
                uint64_t w0, w1, w2;
                long it = 0;
                for (;;) {
                    w0 = ld_pkt(ps);
                    w1 = ld_pkt(ps + 1);
                    w2 = ld_pkt(ps + 2);
                    if ((uint32_t)(w0 >> 32) == tag && (uint32_t)(w1 >> 32) == tag && (uint32_t)(w2 >> 32) == tag)
                        break;
                    if (spin_give_up(it, a.err)) break;
                }
                const double v2 = __longlong_as_double((long long)(((w1 & 0xffffffffull) << 32) | (w0 & 0xffffffffull)));
                const int r2 = (int)(uint32_t)w2;
                if (better(v2, r2, gv, gr)) { gv = v2; gr = r2; gs = s; }
            }
            const int l = wave_best(gv, gr, gr != kNoRow);
            const int r = l >= 0 ? __builtin_amdgcn_readlane(gr, l) : kNoRow;
            // no usable candidate (non-finite column): a zero pivot in place
            const bool ok = r >= pr && r < a.n;
            double m = 0.0;
            double2 rinv = make_double2(0.0, 0.0);
            if (ok) {
                m = readlane_f64(gv, l);
                constexpr int PL = NW / 64;  // pivot-row words per lane, loaded together
                const uint64_t *pu = cand + (size_t)__builtin_amdgcn_readlane(gs, l) * NWS + lane;
                uint64_t wu[PL];
                long it = 0;
                for (;;) {
                    bool got = true;
#pragma unroll
                    for (int e = 0; e < PL; ++e) {
                        wu[e] = ld_pkt(pu + 64 * e);
                        got = got && (uint32_t)(wu[e] >> 32) == tag;
                    }
                    if (got) break;
                    if (spin_give_up(it, a.err)) break;
                }
#pragma unroll
                for (int e = 0; e < PL; ++e) ((uint32_t *)s_u)[lane + 64 * e] = (uint32_t)wu[e];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const V p = s_u[j];  // written by this wave above
                if (m != 0.0) rinv = crecip((double)p.x, (double)p.y);
            }
            if (lane == 0) {
                s_gv = m;
                s_gr = ok ? r : pr;
                s_rinv = rinv;
            }
        }
        __syncthreads();
        const double gv = s_gv;
        const int gr = s_gr;

        // 5. interchange positions k+j and gr, scale column j, rank-1 update
        const double2 rinv = s_rinv;
        if (tid == 0) s_piv[j] = gr;
        if (tid == 0 && gv == 0.0 && s_zero < 0) s_zero = pr;
        if (lr == gr) lr = pr;
        else if (lr == pr) lr = gr;
        const bool act = gv != 0.0 && valid && lr > pr;
        T lre = 0, lim = 0;
        if (c == cj) {
            if (act) {
                const double2 l = mul_c((double)nxr, (double)nxi, rinv.x, rinv.y);
                lre = (T)l.x;
                lim = (T)l.y;
            }
            if (TPR > 1) s_l[rb * 64 + lane] = V{lre, lim};
        }
        if (TPR > 1) {
            __syncthreads();
            if (c != cj) {
                const V l = s_l[rb * 64 + lane];
                lre = l.x;
                lim = l.y;
            }
        }
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const int col = c * W + i;  // uniform
            if (col == j) {             // the multiplier replaces column j
                if (act) {
                    re[i] = lre;
                    im[i] = lim;
                }
            } else if (col > j) {
                if (sizeof(T) == 4 || act) {  // as in k_panel
                    const V u = s_u[col];
                    re[i] = sub_mul_re(re[i], lre, lim, u.x, u.y);
                    im[i] = sub_mul_im(im[i], lre, lim, u.x, u.y);
                }
                if (col == j + 1) {
                    nxr = re[i];
                    nxi = im[i];
                }
            }
            // keep the scheduler from hoisting every column's pivot-row load at once
            if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
    }

    // each row to its final position
#pragma unroll
    for (int i = 0; i < W; ++i)
        if (valid) Ab[lr + (size_t)(k + c * W + i) * a.lda] = V{re[i], im[i]};
    __syncthreads();  // s_piv complete
    if (w == 0 && tid < NB) a.ipiv[(size_t)b * a.strideP + k + tid] = s_piv[tid] + 1;
    if (w == 0 && tid == 0 && s_zero >= 0 && a.info[b] == 0) a.info[b] = s_zero + 1;
    if (w == 0 && wave == 0) panel_perm(k, lane, s_piv, X.perm(xm, a.pslot));
}

// ---------------------------------------------------------------------------
// Row interchanges outside the panel and U12 = L11^{-1} A12.  Tiles of CB
// columns, three kinds by tile index:
//   [0, ntl)           columns [c_l0, c_l1): interchanges only (to the left)
//   [ntl, ntl+ntr)     columns [c_tr0, c_tr1): interchanges (if do_swap) and
//                      the triangular solve of rows k..k+NB-1
//   [ntl+ntr, ...)     columns [c_sw0, n): interchanges only (columns whose
//                      rows k..k+NB-1 still await earlier panels' updates)
struct SwapArgs {
    int n, k, slots, pslot, c_l0, c_l1, ntl, ntr, c_tr0, c_tr1, c_sw0, do_swap;
    const int *nmem;  // per matrix index: its own size (identity beyond), or null
};

// A wave owns CB / 4 columns, lane = row slot: slots t < NB are rows k + t (one
// contiguous run per column: coalesced), the others the rows from below the
// panel that take part; a column's loads all come before its stores in the same
// wave, so no barrier separates them.  Interchange-only tiles move the slots
// that change; solved tiles keep the new top rows in registers and solve there:
// step j broadcasts x_j by lane reads and takes column j of L11 from LDS (packed
// by columns: consecutive lanes, consecutive entries), without barriers, and
// the rows are stored once.  The arithmetic and its order are a forward
// substitution's.  What a small launch costs is this chain of 63 steps and the
// memory latencies before and after it, a large one moving the rows.  Against
// tiles solved with a barrier per step, per launch: 28 -> 14 us (N = 512), 64 ->
// 35 us (12 x 4096), 37 -> 20 us (2 x 8192), 135 -> 65 us (16 x 8192), pivots near
// the diagonal; 346 -> 302 us (16 x 8192, random pivots).
template <typename T, int CB>
__global__ __launch_bounds__(256) void k_swap_trsm(typename CT<T>::V *A, int lda, int64_t strideA, SwapArgs a,
                                                   char *xbuf, const int *bidx)
{
    using V = typename CT<T>::V;
    constexpr int CW = CB / 4;  // columns per wave
    const int bl = blockIdx.y, tile = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = bidx ? bidx[bl] : bl;
    const int n = a.n, k = a.k;
    V *Ab = A + (size_t)b * strideA;
    const XLayout<V> X(a.slots);
    char *xm = xbuf + (size_t)bl * X.mat_bytes;

    const bool trsm = tile >= a.ntl && tile < a.ntl + a.ntr;
    const int c0 = tile < a.ntl ? a.c_l0 + tile * CB : trsm ? a.c_tr0 + (tile - a.ntl) * CB
                                                   : a.c_sw0 + (tile - a.ntl - a.ntr) * CB;
    const int cend = tile < a.ntl ? a.c_l1 : trsm ? a.c_tr1 : n;
    // beyond the member's own size: no interchanges (its panel was the
    // identity) and zero blocks right of it (their solve changes nothing)
    if (a.nmem && (k >= a.nmem[b] || c0 >= a.nmem[b])) return;

    int src0 = k + lane, src1 = 0, dst1 = 0;
    bool ex = false;
    if (a.do_swap) {
        const int *pm = X.perm(xm, a.pslot);
        const int *rows = pm + 1, *src = pm + 1 + 2 * NB;
        ex = NB + lane < pm[0];
        src0 = src[lane];
        if (ex) {
            src1 = src[NB + lane];
            dst1 = rows[NB + lane];
        }
    }
    const bool move0 = trsm || src0 != k + lane;
    V top[CW], ext[CW];
#pragma unroll
    for (int q = 0; q < CW; ++q) {
        const int col = c0 + wave * CW + q;
        const V *Ac = Ab + (size_t)col * lda;
        top[q] = ext[q] = V{0, 0};
        if (col < cend && move0) top[q] = Ac[src0];
        if (col < cend && ex) ext[q] = Ac[src1];
    }
    __shared__ V s_l[NB * (NB - 1) / 2];  // strictly lower part of L11, column by column
    auto lidx = [](int i, int j) { return j * (2 * NB - 1 - j) / 2 + (i - j - 1); };
    if (trsm) {
        for (int j = wave; j < NB - 1; j += 4)
            if (lane > j) s_l[lidx(lane, j)] = Ab[(k + lane) + (size_t)(k + j) * lda];
    }
#pragma unroll
    for (int q = 0; q < CW; ++q) {
        const int col = c0 + wave * CW + q;
        V *Ac = Ab + (size_t)col * lda;
        if (col < cend && ex) Ac[dst1] = ext[q];
        if (col < cend && !trsm && move0) Ac[k + lane] = top[q];
    }
    if (!trsm) return;
    __syncthreads();
#pragma unroll 8
    for (int j = 0; j < NB - 1; ++j) {
        V xj[CW];
#pragma unroll
        for (int q = 0; q < CW; ++q) xj[q] = V{readlane_t(top[q].x, j), readlane_t(top[q].y, j)};
        if (lane > j) {
            const V l = s_l[lidx(lane, j)];
#pragma unroll
            for (int q = 0; q < CW; ++q)
                top[q] = V{sub_mul_re(top[q].x, xj[q].x, xj[q].y, l.x, l.y),
                           sub_mul_im(top[q].y, xj[q].x, xj[q].y, l.x, l.y)};
        }
    }
#pragma unroll
    for (int q = 0; q < CW; ++q) {
        const int col = c0 + wave * CW + q;
        if (col < cend) Ab[(k + lane) + (size_t)col * lda] = top[q];
    }
}

// ---------------------------------------------------------------------------
// Block update  C (M x N) -= A (M x K) * B (K x N)  on the matrix cores.
//
// Both kernels issue the MFMA on the transposed problem, C^T = B^T A^T:
// MFMA rows are columns of C and MFMA columns are rows of C, so each
// accumulator register of a lane maps to a run of consecutive rows of one
// column of C and the read-modify-write of C is coalesced.  Complex products
// take three real products (below).  K is walked in chunks staged through
// LDS (8 for complex128, 16 for complex64); the next chunk is fetched from
// global memory into registers while the current one is multiplied.  The entries
// of C are loaded several at a time before any is stored (out-of-range lanes
// load the last row or column): one by one, each under its own condition, every
// one waited for memory in turn, most of a K = 64 update (N = 8192: complex64 400
// -> 310 us, split-BF16x3 437 -> 249 us; complex128 at N = 2048 43 -> 41).
//
// Tiles are dealt to the XCDs in contiguous runs (workgroup ids go to the 8
// XCDs round-robin) and ordered in groups of row tiles (tile_coords), so the
// tiles an XCD runs at once share their L and U blocks in its L2.

// C = A[r0.., c0..] (mrows x ncols) -= A[r0.., kk..kk+K) * A[kk..kk+K, c0..); K a multiple of 64.
struct GemmArgs {
    int r0, c0, mrows, ncols, kk, K;
    const int *nmem;  // per matrix index: its own size (identity beyond, so its updates there are zero), or null
};

// Tile of workgroup g out of T, grouped per XCD; >= T means "no tile".
__device__ inline int xcd_tile(int g, int T)
{
    const int per = (T + 7) / 8;
    return (g % 8) * per + g / 8;
}

inline int xcd_grid(int T) { return 8 * ((T + 7) / 8); }

// Tile t (of TI x TJ) -> (row tile, column tile), in groups of kGroupM row
// tiles: consecutive t walk down a group's rows, then across its columns.
// With the contiguous per-XCD runs of xcd_tile, the 64 tiles an XCD runs at
// once cover about 8 row blocks x 8 column blocks, so their L and U blocks
// are shared through that XCD's L2 instead of each tile streaming its own.
constexpr int kGroupM = 8;
__device__ inline void tile_coords(int t, int TI, int TJ, int &ti, int &tj)
{
    const int per = kGroupM * TJ;
    const int g = t / per, r0 = g * kGroupM;
    const int rows = (TI - r0 < kGroupM) ? TI - r0 : kGroupM;
    const int u = t - g * per;
    ti = r0 + u % rows;
    tj = u / rows;
}

// complex128 with three real products per complex product (Gauss): over the
// K terms, P = sum Br Ar, Q = sum Bi Ai and S = sum (Br + Bi)(Ar + Ai), so
// Re(LU) = P - Q and Im(LU) = S - P - Q.  Three accumulators instead of two
// make the wave tile 32 x 32 (2 x 2 tiles of v_mfma_f64_16x16x4f64, lane l
// holding srcA[l%16][l/16], srcB[l/16][l%16] and D[l/16 + 4*v][l%16]);
// workgroup tile 64 x 64.  Against four products this takes a quarter fewer
// MFMA cycles per update.  The error bound per entry is that of the
// four-product form with |a||b| replaced by (|Ar| + |Ai|)(|Br| + |Bi|), at
// most twice as large.
// K is staged through LDS in chunks of 8: the smaller chunk's prefetch registers
// keep the kernel at three waves per SIMD, which hides the LDS and global
// latency better than two waves with chunks of 16 (83 % against 78 % of the
// FP64 matrix-core peak issued at K = 512, N = 8192).  Two chunks are in flight
// in registers (the next to stage and the one after): 168 VGPRs, four dwords of
// tile bookkeeping spilled outside the loop, 1 % faster than one chunk.
constexpr int GZ_BM = 64, GZ_BN = 64, GZ_KC = 8;

__global__ __launch_bounds__(256, 3) void k_gemm_f64(double2 *Abase, int lda, int64_t strideA, GemmArgs g,
                                                     const int *bidx, int TI, int TJ)
{
    const int t = xcd_tile(blockIdx.x, TI * TJ);
    if (t >= TI * TJ) return;
    const int b = bidx ? bidx[blockIdx.z] : (int)blockIdx.z;
    double2 *M = Abase + (size_t)b * strideA;
    const int mrows = g.mrows, ncols = g.ncols, K = g.K;
    int ti, tj;
    tile_coords(t, TI, TJ, ti, tj);
    const int i0 = ti * GZ_BM, j0 = tj * GZ_BN;
    if (g.nmem && (g.r0 + i0 >= g.nmem[b] || g.c0 + j0 >= g.nmem[b])) return;
    const double2 *A = M + g.r0 + (size_t)g.kk * lda;  // L block
    const double2 *B = M + g.kk + (size_t)g.c0 * lda;  // U block
    double2 *C = M + g.r0 + (size_t)g.c0 * lda;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;

    constexpr int EA = GZ_KC / 4, BJS = 256 / GZ_KC, EB = GZ_BN / BJS;
    __shared__ double2 sA[GZ_KC][GZ_BM + 1];
    __shared__ double2 sB[GZ_KC][GZ_BN + 1];
    // two chunks in flight in registers: the one to stage next and the one after
    double2 pa0[EA], pb0[EB], pa1[EA], pb1[EB];
    // chunk elements moved by this thread: L rows ai, k = ak + 4e; U k = bk, columns bj + BJS e
    const int ai = tid % GZ_BM, ak = tid / GZ_BM;
    const int bk = tid % GZ_KC, bj = tid / GZ_KC;
    const bool arow = i0 + ai < mrows;
    auto fetch = [&](int kc, double2 *pa, double2 *pb) {
        const double2 *pA = A + (i0 + ai) + (size_t)(kc + ak) * lda;
#pragma unroll
        for (int e = 0; e < EA; ++e) pa[e] = arow ? pA[(size_t)(4 * e) * lda] : double2{0.0, 0.0};
        const double2 *pB = B + (kc + bk) + (size_t)(j0 + bj) * lda;
#pragma unroll
        for (int e = 0; e < EB; ++e) pb[e] = (j0 + bj + BJS * e < ncols) ? pB[(size_t)(BJS * e) * lda] : double2{0.0, 0.0};
    };
    auto stash = [&](const double2 *pa, const double2 *pb) {
#pragma unroll
        for (int e = 0; e < EA; ++e) sA[ak + 4 * e][ai] = pa[e];
#pragma unroll
        for (int e = 0; e < EB; ++e) sB[bk][bj + BJS * e] = pb[e];
    };
    v4d P[2][2], Q[2][2], S[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) { P[x][y] = v4d{0, 0, 0, 0}; Q[x][y] = P[x][y]; S[x][y] = P[x][y]; }
    auto compute = [&]() {
#pragma unroll
        for (int ks = 0; ks < GZ_KC; ks += 4) {
            const int kk = ks + lane / 16;
            double2 bv[2], av[2];
            double bs[2], as[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                bv[q] = sB[kk][wj + q * 16 + lane % 16];
                av[q] = sA[kk][wi + q * 16 + lane % 16];
                bs[q] = bv[q].x + bv[q].y;
                as[q] = av[q].x + av[q].y;
            }
#pragma unroll
            for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                for (int ti = 0; ti < 2; ++ti) P[tj][ti] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[tj].x, av[ti].x, P[tj][ti], 0, 0, 0);
#pragma unroll
            for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                for (int ti = 0; ti < 2; ++ti) Q[tj][ti] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[tj].y, av[ti].y, Q[tj][ti], 0, 0, 0);
#pragma unroll
            for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                for (int ti = 0; ti < 2; ++ti) S[tj][ti] = __builtin_amdgcn_mfma_f64_16x16x4f64(bs[tj], as[ti], S[tj][ti], 0, 0, 0);
        }
    };

    // K is a multiple of 2 chunks: the loop takes two chunks per trip, chunk
    // kc from LDS while chunk kc + GZ_KC waits in pa1/pb1 and kc + 2 GZ_KC loads
    fetch(0, pa0, pb0);
    stash(pa0, pb0);
    fetch(GZ_KC, pa1, pb1);
    __syncthreads();
    for (int kc = 0; kc < K; kc += 2 * GZ_KC) {
        if (kc + 2 * GZ_KC < K) fetch(kc + 2 * GZ_KC, pa0, pb0);
        compute();
        __syncthreads();
        stash(pa1, pb1);
        __syncthreads();
        if (kc + 3 * GZ_KC < K) fetch(kc + 3 * GZ_KC, pa1, pb1);
        compute();
        if (kc + 2 * GZ_KC < K) {
            __syncthreads();
            stash(pa0, pb0);
            __syncthreads();
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) {
        double2 c[2][4];
#pragma unroll
        for (int ti = 0; ti < 2; ++ti)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                c[ti][v] = C[min(i0 + wi + ti * 16 + lane % 16, mrows - 1) +
                             (size_t)min(j0 + wj + tj * 16 + lane / 16 + 4 * v, ncols - 1) * lda];
#pragma unroll
        for (int ti = 0; ti < 2; ++ti)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int gi = i0 + wi + ti * 16 + lane % 16;
                const int gj = j0 + wj + tj * 16 + (lane / 16) + 4 * v;
                const double p = P[tj][ti][v], q = Q[tj][ti][v];
                c[ti][v].x -= p - q;
                c[ti][v].y -= S[tj][ti][v] - p - q;
                if (gi < mrows && gj < ncols) C[gi + (size_t)gj * lda] = c[ti][v];
            }
    }
}

// The complex128 update of launches with too few 64 x 64 tiles to fill the device
// (small matrices, the narrow updates inside an outer block): the same products
// in the same order (the same bits) on tiles of 32 x 32, one 16 x 16 tile per wave,
// so four times as many workgroups share the work.  Such a launch is a chain of
// latencies: both operands' first two chunks of 32 (all of K = 64) and the C tile
// are loaded at once at the start, and a chunk needs one barrier.
constexpr int GS_B = 32, GS_KC = 32;

__global__ __launch_bounds__(256, 2) void k_gemm_f64_small(double2 *Abase, int lda, int64_t strideA, GemmArgs g,
                                                           const int *bidx, int TI, int TJ)
{
    const int t = xcd_tile(blockIdx.x, TI * TJ);
    if (t >= TI * TJ) return;
    const int b = bidx ? bidx[blockIdx.z] : (int)blockIdx.z;
    double2 *M = Abase + (size_t)b * strideA;
    const int mrows = g.mrows, ncols = g.ncols, K = g.K;
    int ti, tj;
    tile_coords(t, TI, TJ, ti, tj);
    const int i0 = ti * GS_B, j0 = tj * GS_B;
    if (g.nmem && (g.r0 + i0 >= g.nmem[b] || g.c0 + j0 >= g.nmem[b])) return;
    const double2 *A = M + g.r0 + (size_t)g.kk * lda;  // L block
    const double2 *B = M + g.kk + (size_t)g.c0 * lda;  // U block
    double2 *C = M + g.r0 + (size_t)g.c0 * lda;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 16, wj = (wave >> 1) * 16;

    // two buffers: a chunk is staged while the other is still read
    __shared__ double2 sA[2][GS_KC][GS_B + 1];
    __shared__ double2 sB[2][GS_KC][GS_B + 1];
    double2 pa[2][4], pb[2][4];
    // chunk elements moved by this thread: L row ai, k = ak + 8e; U k = bk, columns bj + 8e
    const int ai = tid % GS_B, ak = tid / GS_B, bk = tid % GS_KC, bj = tid / GS_KC;
    const bool arow = i0 + ai < mrows;
    auto fetch = [&](int kc, double2 *a, double2 *u) {
        const double2 *pA = A + (i0 + ai) + (size_t)(kc + ak) * lda;
        const double2 *pB = B + (kc + bk) + (size_t)(j0 + bj) * lda;
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = arow ? pA[(size_t)(8 * e) * lda] : double2{0.0, 0.0};
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = (j0 + bj + 8 * e < ncols) ? pB[(size_t)(8 * e) * lda] : double2{0.0, 0.0};
    };
    auto stash = [&](int buf, const double2 *a, const double2 *u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sA[buf][ak + 8 * e][ai] = a[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) sB[buf][bk][bj + 8 * e] = u[e];
    };
    fetch(0, pa[0], pb[0]);
    if (GS_KC < K) fetch(GS_KC, pa[1], pb[1]);
    const int gi = i0 + wi + lane % 16, gj = j0 + wj + lane / 16;
    double2 c[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
        c[v] = gi < mrows && gj + 4 * v < ncols ? C[gi + (size_t)(gj + 4 * v) * lda] : double2{0.0, 0.0};

    v4d P = v4d{0, 0, 0, 0}, Q = P, S = P;
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < GS_KC; ks += 4) {
            const int kk = ks + lane / 16;
            const double2 bv = sB[buf][kk][wj + lane % 16], av = sA[buf][kk][wi + lane % 16];
            P = __builtin_amdgcn_mfma_f64_16x16x4f64(bv.x, av.x, P, 0, 0, 0);
            Q = __builtin_amdgcn_mfma_f64_16x16x4f64(bv.y, av.y, Q, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f64_16x16x4f64(bv.x + bv.y, av.x + av.y, S, 0, 0, 0);
        }
    };
    // K is a multiple of two chunks; a buffer is written again only after the
    // barrier that follows its last reads
    for (int kc = 0; kc < K; kc += 2 * GS_KC) {
        stash(0, pa[0], pb[0]);
        if (kc + 2 * GS_KC < K) fetch(kc + 2 * GS_KC, pa[0], pb[0]);
        __syncthreads();
        compute(0);
        stash(1, pa[1], pb[1]);
        if (kc + 3 * GS_KC < K) fetch(kc + 3 * GS_KC, pa[1], pb[1]);
        __syncthreads();
        compute(1);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (gi < mrows && gj + 4 * v < ncols) {
            const double p = P[v], q = Q[v];
            C[gi + (size_t)(gj + 4 * v) * lda] = double2{c[v].x - (p - q), c[v].y - (S[v] - p - q)};
        }
}

// complex64 with three real products per complex product, as k_gemm_f64:
// P = sum Br Ar, Q = sum Bi Ai, S = sum (Br + Bi)(Ar + Ai).  Workgroup tile
// 128 x 64, four waves of 64 x 32 (2 x 1 tiles of v_mfma_f32_32x32x2f32).
// Lane l holds srcA[l%32][l/32], srcB[l/32][l%32] and
// D[8*(v/4)+4*(l/32)+v%4][l%32].
constexpr int GC_BM = 128, GC_BN = 64, GC_KC = 16;

__global__ __launch_bounds__(256, 2) void k_gemm_f32(float2 *Abase, int lda, int64_t strideA, GemmArgs g,
                                                     const int *bidx, int TI, int TJ)
{
    const int t = xcd_tile(blockIdx.x, TI * TJ);
    if (t >= TI * TJ) return;
    const int b = bidx ? bidx[blockIdx.z] : (int)blockIdx.z;
    float2 *M = Abase + (size_t)b * strideA;
    const int mrows = g.mrows, ncols = g.ncols, K = g.K;
    int ti, tj;
    tile_coords(t, TI, TJ, ti, tj);
    const int i0 = ti * GC_BM, j0 = tj * GC_BN;
    if (g.nmem && (g.r0 + i0 >= g.nmem[b] || g.c0 + j0 >= g.nmem[b])) return;
    const float2 *A = M + g.r0 + (size_t)g.kk * lda;
    const float2 *B = M + g.kk + (size_t)g.c0 * lda;
    float2 *C = M + g.r0 + (size_t)g.c0 * lda;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 64, wj = (wave >> 1) * 32;

    __shared__ float2 sA[GC_KC][GC_BM + 2];
    __shared__ float2 sB[GC_KC][GC_BN + 2];
    float2 pa[8], pb[4];
    // chunk elements moved by this thread: L rows ai, k = ak + 2e; U k = bk, columns bj + 16e
    const int ai = tid % GC_BM, ak = tid / GC_BM;
    const int bk = tid % GC_KC, bj = tid / GC_KC;
    const bool arow = i0 + ai < mrows;
    auto fetch = [&](int kc) {
        const float2 *pA = A + (i0 + ai) + (size_t)(kc + ak) * lda;
#pragma unroll
        for (int e = 0; e < 8; ++e) pa[e] = arow ? pA[(size_t)(2 * e) * lda] : float2{0.f, 0.f};
        const float2 *pB = B + (kc + bk) + (size_t)(j0 + bj) * lda;
#pragma unroll
        for (int e = 0; e < 4; ++e) pb[e] = (j0 + bj + 16 * e < ncols) ? pB[(size_t)(16 * e) * lda] : float2{0.f, 0.f};
    };
    auto stash = [&]() {
#pragma unroll
        for (int e = 0; e < 8; ++e) sA[ak + 2 * e][ai] = pa[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) sB[bk][bj + 16 * e] = pb[e];
    };
    v16f P[2], Q[2], S[2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int v = 0; v < 16; ++v) { P[x][v] = 0.f; Q[x][v] = 0.f; S[x][v] = 0.f; }

    fetch(0);
    stash();
    __syncthreads();
    for (int kc = 0; kc < K; kc += GC_KC) {
        if (kc + GC_KC < K) fetch(kc + GC_KC);
#pragma unroll
        for (int ks = 0; ks < GC_KC; ks += 2) {
            const int kk = ks + lane / 32;
            const float2 bv = sB[kk][wj + lane % 32];
            const float bs = bv.x + bv.y;
            float2 av[2];
            float as[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                av[q] = sA[kk][wi + q * 32 + lane % 32];
                as[q] = av[q].x + av[q].y;
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) P[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv.x, av[q].x, P[q], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 2; ++q) Q[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv.y, av[q].y, Q[q], 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 2; ++q) S[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(bs, as[q], S[q], 0, 0, 0);
        }
        if (kc + GC_KC < K) {
            __syncthreads();
            stash();
            __syncthreads();
        }
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) {  // eight elements at a time: 168 VGPRs, three waves per SIMD
        const int q = h / 2, v0 = h % 2 * 8;
        float2 c[8];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = v0; v < v0 + 8; ++v)
            c[v - v0] = C[min(i0 + wi + q * 32 + lane % 32, mrows - 1) +
                          (size_t)min(j0 + wj + 8 * (v / 4) + 4 * (lane / 32) + (v % 4), ncols - 1) * lda];
#pragma unroll
        for (int v = v0; v < v0 + 8; ++v) {
            const int gi = i0 + wi + q * 32 + lane % 32;
            const int gj = j0 + wj + 8 * (v / 4) + 4 * (lane / 32) + (v % 4);
            const float p = P[q][v], r = Q[q][v];
            c[v - v0].x -= p - r;
            c[v - v0].y -= S[q][v] - p - r;
            if (gi < mrows && gj < ncols) C[gi + (size_t)gj * lda] = c[v - v0];
        }
    }
}

// complex64 with split-BF16x3 products: every FP32 operand x is split into
// bf16 hi = rn(x) and lo = rn(x - hi), and each real product X*Y is taken as
// Xhi*Yhi + Xhi*Ylo + Xlo*Yhi on v_mfma_f32_32x32x16_bf16 with FP32
// accumulation (relative error about 2^-16 per product instead of 2^-24).
// Workgroup tile 128 x 128, four waves of 64 x 64 (2 x 2 MFMA tiles), K in
// chunks of 16.  Lane l holds srcA[l%32][8*(l/32)+i], srcB[8*(l/32)+i][l%32]
// (i = 0..7) and D[8*(v/4)+4*(l/32)+v%4][l%32].  The chunk is staged in LDS as
// four bf16 planes (re hi, re lo, im hi, im lo) with k contiguous per row of L
// and per column of U, so each operand is one 16-byte LDS read.  A row is 32
// bytes, two 16-byte halves, stored swapped in rows 8-15 of every 16 (an XOR
// swizzle instead of padding), so rows 0 and 8 of a pass no longer share banks
// (bank-conflict cycles 43 -> 20 % of the LDS's active cycles).  Two LDS buffers
// (64 KiB, two workgroups per CU): while the waves multiply one chunk they
// split and store the next (already in registers) into the other buffer and
// load the one after, with one barrier per chunk.  Rows and columns beyond the
// update load the last one's values (their products reach no stored entry), so
// the loads need no condition and a column's eight elements come as four 16-byte
// loads: N = 8192, K = 512: 905 -> 742 us.  A chunk's products are issued before
// the next one's splitting, which runs beside them: 742 -> 690 (alone on its CU a
// workgroup's chunk takes 1.35 us instead of 1.75).  Eight lanes per column of U,
// two k each, whole lines per load but 4-byte LDS stores: 722.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(8)));
constexpr int GB_BM = 128, GB_BN = 128, GB_KC = 16;

// Two values (consecutive k) at once: hi and lo pairs as words.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ inline void split_bf16(float x, float y, unsigned &hi, unsigned &lo)
{
    hi = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x, y}), bf16x2));
    const float hx = __builtin_bit_cast(float, hi << 16), hy = __builtin_bit_cast(float, hi & 0xffff0000u);
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x - hx, y - hy}), bf16x2));
}

// k offset (bf16) of half h (0: k 0-7, 1: k 8-15) of LDS row r of a chunk
__device__ inline int b3_half(int r, int h) { return 8 * (h ^ ((r >> 3) & 1)); }

__device__ inline bf16x8 neg_bf16x8(bf16x8 v)
{
    u32x4 u = __builtin_bit_cast(u32x4, v);
    u ^= 0x80008000u;
    return __builtin_bit_cast(bf16x8, u);
}

__global__ __launch_bounds__(256, 2) void k_gemm_b3(float2 *Abase, int lda, int64_t strideA, GemmArgs g,
                                                    const int *bidx, int TI, int TJ)
{
    const int t = xcd_tile(blockIdx.x, TI * TJ);
    if (t >= TI * TJ) return;
    const int b = bidx ? bidx[blockIdx.z] : (int)blockIdx.z;
    float2 *M = Abase + (size_t)b * strideA;
    const int mrows = g.mrows, ncols = g.ncols, K = g.K;
    int ti, tj;
    tile_coords(t, TI, TJ, ti, tj);
    const int i0 = ti * GB_BM, j0 = tj * GB_BN;
    if (g.nmem && (g.r0 + i0 >= g.nmem[b] || g.c0 + j0 >= g.nmem[b])) return;
    const float2 *A = M + g.r0 + (size_t)g.kk * lda;  // L block
    const float2 *B = M + g.kk + (size_t)g.c0 * lda;  // U block
    float2 *C = M + g.r0 + (size_t)g.c0 * lda;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 64, wj = (wave >> 1) * 64;

    // [buffer][plane: 0 re hi, 1 re lo, 2 im hi, 3 im lo][row][k]
    __shared__ __attribute__((aligned(16))) __bf16 sL[2][4][GB_BM][GB_KC];
    __shared__ __attribute__((aligned(16))) __bf16 sU[2][4][GB_BN][GB_KC];
    // chunk elements moved by this thread: 8 consecutive k of one row of L and of one column of U
    const int lr = tid % GB_BM, lh = tid / GB_BM;  // L: row lr, k = 8*lh + e
    const int uc = tid / 2, uh = tid % 2;           // U: column uc, k = 8*uh + e
    const float2 *pA = A + min(i0 + lr, mrows - 1) + (size_t)(8 * lh) * lda;
    const float2 *pB = B + 8 * uh + (size_t)min(j0 + uc, ncols - 1) * lda;
    float2 pa[8];
    f32x4 pb[4];  // two elements of U each; an element's alignment is all that lda promises
    auto fetch = [&](int kc) {
#pragma unroll
        for (int e = 0; e < 8; ++e) pa[e] = pA[(size_t)(kc + e) * lda];
#pragma unroll
        for (int e = 0; e < 4; ++e) pb[e] = *(const f32x4 *)(pB + kc + 2 * e);
    };
    auto stash = [&](int buf) {
        u32x4 v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            unsigned h, l;
            split_bf16(pa[2 * e].x, pa[2 * e + 1].x, h, l);
            v[0][e] = h;
            v[1][e] = l;
            split_bf16(pa[2 * e].y, pa[2 * e + 1].y, h, l);
            v[2][e] = h;
            v[3][e] = l;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) *(u32x4 *)&sL[buf][q][lr][b3_half(lr, lh)] = v[q];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            unsigned h, l;
            split_bf16(pb[e][0], pb[e][2], h, l);
            v[0][e] = h;
            v[1][e] = l;
            split_bf16(pb[e][1], pb[e][3], h, l);
            v[2][e] = h;
            v[3][e] = l;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) *(u32x4 *)&sU[buf][q][uc][b3_half(uc, uh)] = v[q];
    };
    v16f accR[2][2], accI[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 16; ++v) { accR[x][y][v] = 0.f; accI[x][y][v] = 0.f; }

    auto compute = [&](int buf) {
        // U operands (MFMA rows = columns of C), L operands (MFMA columns = rows of C)
        bf16x8 ur[2][2], ui[2][2], un[2][2], lre[2][2], lim[2][2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int cj = wj + q * 32 + lane % 32, ri = wi + q * 32 + lane % 32;
            const int ku = b3_half(cj, lane / 32), kl = b3_half(ri, lane / 32);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                ur[q][h] = *(const bf16x8 *)&sU[buf][0 + h][cj][ku];
                ui[q][h] = *(const bf16x8 *)&sU[buf][2 + h][cj][ku];
                un[q][h] = neg_bf16x8(ui[q][h]);
                lre[q][h] = *(const bf16x8 *)&sL[buf][0 + h][ri][kl];
                lim[q][h] = *(const bf16x8 *)&sL[buf][2 + h][ri][kl];
            }
        }
        // split terms (hi,hi), (hi,lo), (lo,hi); real and imaginary accumulators alternate
#pragma unroll
        for (int term = 0; term < 3; ++term) {
            const int hu = term == 2 ? 1 : 0, hl = term == 1 ? 1 : 0;
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    accR[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ur[x][hu], lre[y][hl], accR[x][y], 0, 0, 0);
                    accI[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ur[x][hu], lim[y][hl], accI[x][y], 0, 0, 0);
                }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    accR[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(un[x][hu], lim[y][hl], accR[x][y], 0, 0, 0);
                    accI[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ui[x][hu], lre[y][hl], accI[x][y], 0, 0, 0);
                }
        }
    };

    fetch(0);
    stash(0);
    fetch(GB_KC);  // K is a multiple of 64
    __syncthreads();
    int buf = 0;
    for (int kc = 0; kc + GB_KC < K; kc += GB_KC, buf ^= 1) {
        compute(buf);
        stash(buf ^ 1);
        fetch(min(kc + 2 * GB_KC, K - GB_KC));
        __syncthreads();
    }
    compute(buf);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            float2 c[16];
#pragma unroll
            for (int v = 0; v < 16; ++v)
                c[v] = C[min(i0 + wi + y * 32 + lane % 32, mrows - 1) +
                         (size_t)min(j0 + wj + x * 32 + 8 * (v / 4) + 4 * (lane / 32) + (v % 4), ncols - 1) * lda];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int gi = i0 + wi + y * 32 + lane % 32;
                const int gj = j0 + wj + x * 32 + 8 * (v / 4) + 4 * (lane / 32) + (v % 4);
                c[v].x -= accR[x][y][v];
                c[v].y -= accI[x][y][v];
                if (gi < mrows && gj < ncols) C[gi + (size_t)gj * lda] = c[v];
            }
        }
}

// Launches the interchanges and solves of one panel for m matrices; sa without
// its tile counts.  Tiles of 8 columns (two per wave) shorten the chain of a
// launch that leaves the device idle, tiles of 16 read L11 half as often: 14.4
// against 17.5 us per launch at N = 512, 20.3 against 22.7 at 2 x 8192 (512 wide
// tiles and fewer per matrix), 75 against 65 at 16 x 8192.
template <typename T>
void launch_swap(const wm_ctx *ctx, SwapArgs sa, typename CT<T>::V *A, int lda, int64_t strideA, char *xbuf,
                 const int *bidx, int m, hipStream_t s)
{
    const int left = sa.do_swap ? std::max(0, sa.c_l1 - sa.c_l0) : 0, solve = std::max(0, sa.c_tr1 - sa.c_tr0),
              right = sa.do_swap ? std::max(0, sa.n - sa.c_sw0) : 0;
    auto tiles = [&](int cb) {
        sa.ntl = (left + cb - 1) / cb;
        sa.ntr = (solve + cb - 1) / cb;
        return sa.ntl + sa.ntr + (right + cb - 1) / cb;
    };
    const int wide = tiles(16);
    if (wide == 0) return;
    if ((int64_t)wide * m <= 4 * ctx->num_cu) {
        const int t = tiles(8);
        hipLaunchKernelGGL((k_swap_trsm<T, 8>), dim3(t, m), dim3(256), 0, s, A, lda, strideA, sa, xbuf, bidx);
    } else {
        hipLaunchKernelGGL((k_swap_trsm<T, 16>), dim3(wide, m), dim3(256), 0, s, A, lda, strideA, sa, xbuf, bidx);
    }
}

// Most 64 x 64 tiles of a complex128 update that runs on tiles of 32 x 32: 14 -> 6 us
// with 49 tiles, 24.5 -> 22.0 with 361, 31.0 -> 30.9 with 529 (K = 64); 36 -> 12 us with
// 16, 41.7 -> 37.4 with 256, 62.5 -> 61.5 with 400 (K = 256).
constexpr int64_t kSmallTiles = 512;

// Launches C -= L U for nb_ matrices, C = A[r0.., c0..] (mrows x ncols),
// L = A[r0.., kk..kk+K), U = A[kk..kk+K, c0..).  gk: 8 complex128, 4 complex64,
// 2 complex64 with split-BF16x3 products.
void launch_gemm(int gk, void *A, int lda, int64_t strideA, const GemmArgs &g, int nb_, const int *bidx,
                 hipStream_t s)
{
    if (g.mrows <= 0 || g.ncols <= 0 || g.K <= 0) return;
    if (gk == 8) {
        int TI = (g.mrows + GZ_BM - 1) / GZ_BM, TJ = (g.ncols + GZ_BN - 1) / GZ_BN;
        if ((int64_t)TI * TJ * nb_ <= kSmallTiles) {
            TI = (g.mrows + GS_B - 1) / GS_B;
            TJ = (g.ncols + GS_B - 1) / GS_B;
            hipLaunchKernelGGL(k_gemm_f64_small, dim3(xcd_grid(TI * TJ), 1, nb_), dim3(256), 0, s, (double2 *)A, lda,
                               strideA, g, bidx, TI, TJ);
            return;
        }
        hipLaunchKernelGGL(k_gemm_f64, dim3(xcd_grid(TI * TJ), 1, nb_), dim3(256), 0, s, (double2 *)A, lda, strideA,
                           g, bidx, TI, TJ);
    } else if (gk == 4) {
        const int TI = (g.mrows + GC_BM - 1) / GC_BM, TJ = (g.ncols + GC_BN - 1) / GC_BN;
        hipLaunchKernelGGL(k_gemm_f32, dim3(xcd_grid(TI * TJ), 1, nb_), dim3(256), 0, s, (float2 *)A, lda, strideA,
                           g, bidx, TI, TJ);
    } else {
        const int TI = (g.mrows + GB_BM - 1) / GB_BM, TJ = (g.ncols + GB_BN - 1) / GB_BN;
        hipLaunchKernelGGL(k_gemm_b3, dim3(xcd_grid(TI * TJ), 1, nb_), dim3(256), 0, s, (float2 *)A, lda, strideA,
                           g, bidx, TI, TJ);
    }
}

__global__ void k_zero_int(int *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_zero_idx(int *p, const int *idx, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[idx[i]] = 0;
}

__global__ void k_zero_u64(uint64_t *p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_tag_bump(uint32_t *tag, uint32_t inc)
{
    if (threadIdx.x == 0) *tag += inc;
}

__global__ void k_tag_set(uint32_t *tag, uint32_t v)
{
    if (threadIdx.x == 0) *tag = v;
}

// Exchange buffer of at least `bytes` for a factorization that uses `ntags`
// packet tags.  Tags come from the device counter ctx->d_tag, which every launch
// chunk bumps by n (so replays of a captured factorization get fresh tags); the
// host tracks the same count.  The buffer is cleared, and the counter reset,
// when the buffer is (re)allocated and before the counter could wrap, so no
// stale packet can carry a current tag.  A reallocation drops the captured
// factorizations, which hold the old buffer.
int prepare_xbuf(wm_ctx *ctx, size_t bytes, uint64_t ntags, hipStream_t s)
{
    if (ntags > 0x40000000u) {
        set_error("getrf: %llu panel tags in one call", (unsigned long long)ntags);
        return WM_ERR_ARG;
    }
    const size_t had = ctx->ws_lu.bytes;
    WM_TRY(ctx->ws_lu.ensure(bytes));
    const bool fresh = ctx->ws_lu.bytes != had;
    if (fresh) drop_graphs(ctx);
    if (fresh || ctx->panel_tag + ntags + NB > 0xFFFFFFFFull) {
        const size_t nw = ctx->ws_lu.bytes / sizeof(uint64_t);
        hipLaunchKernelGGL(k_zero_u64, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s,
                           (uint64_t *)ctx->ws_lu.ptr, nw);
        hipLaunchKernelGGL(k_tag_set, dim3(1), dim3(64), 0, s, ctx->d_tag, 0u);
        ctx->panel_tag = 0;
    }
    return WM_OK;
}

// The panel kernel with TPR parts per row.
template <typename T, int TPR>
constexpr bool kTall = TPR != (sizeof(T) == 8 ? kTprF64 : kTprF32);
template <typename T, int TPR>
auto panel_kernel()
{
    if constexpr (kTall<T, TPR>) return k_panel_tall<T, TPR>;
    else return k_panel<T, TPR>;
}

template <typename T, int TPR>
int occupancy_panel(int *blocks_per_cu)
{
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, panel_kernel<T, TPR>(), 256, 0);
    if (e != hipSuccess) {
        set_error("occupancy query failed: %s", hipGetErrorString(e));
        return WM_ERR_HIP;
    }
    return WM_OK;
}

// Launch plan of a batched factorization.  All members step through the
// panels together; a panel launch holds as many members as keep every panel
// cluster co-resident at that panel's height (resident / P workgroups), so
// tall panels go in several launches and short ones in one, and each member
// has its own exchange buffer.
struct GetrfPlan {
    int pmax = 0, slots = 0, resident = 0, per_launch = 0;
    size_t xbytes = 0;
};

// Panel workgroups of this context that may be resident at once: the occupancy,
// shared with the other contexts that factor on the device at the same time
// (panel_share), so that every cluster of every concurrent panel launch fits on
// the device together.
template <typename T, int TPR>
int panel_total(wm_ctx *ctx, int *total, int share = 1)
{
    int bpc = 0;
    WM_TRY((occupancy_panel<T, TPR>(&bpc)));
    *total = bpc * ctx->num_cu / share;
    if (ctx->panel_resident_cap > 0 && ctx->panel_resident_cap < *total) *total = ctx->panel_resident_cap;
    return WM_OK;
}

template <typename T, int TPR>
int panel_resident(wm_ctx *ctx, int *resident)
{
    return panel_total<T, TPR>(ctx, resident, std::max(1, ctx->panel_share));
}

template <typename T, int TPR>
int getrf_plan(wm_ctx *ctx, int n, int batch, GetrfPlan *pl)
{
    using V = typename CT<T>::V;
    constexpr int RW = 256 / TPR;
    const int pmax = (n + RW - 1) / RW;
    int resident = 0;
    WM_TRY((panel_resident<T, TPR>(ctx, &resident)));
    if (pmax > resident) {
        set_error("getrf: panel cluster of %d workgroups exceeds %d resident", pmax, resident);
        return WM_ERR_ARG;
    }
    pl->pmax = pmax;
    pl->resident = resident;
    pl->per_launch = std::min(batch, resident / pmax);
    pl->slots = kTall<T, TPR> ? pmax : pmax * (RW / 64);
    pl->xbytes = (size_t)batch * XLayout<V>(pl->slots).mat_bytes;
    return WM_OK;
}

// Enqueues the launches of a planned factorization on s (kernel launches only,
// so the sequence can be captured into a graph).
template <typename T, int TPR>
int getrf_impl(wm_ctx *ctx, const GetrfPlan &pl, int n, typename CT<T>::V *A, int lda, int64_t strideA, int *ipiv,
               int64_t strideP, int batch, int *d_info, const int *d_bidx, hipStream_t s, int gk, int kSub,
               const int *d_nmem, hipStream_t side)
{
    using V = typename CT<T>::V;
    constexpr int RW = 256 / TPR;
    const XLayout<V> X(pl.slots);
    char *xbase = (char *)ctx->ws_lu.ptr;
    const double esz = 2.0 * sizeof(T);
    const int kPanelClass = sizeof(T) == 8 ? K_PANEL : K_PANEL32;
    const int kSwapClass = sizeof(T) == 8 ? K_SWAP : K_SWAP32;
    const int kGemmClass = sizeof(T) == 8 ? K_GEMM : gk == 2 ? K_GEMMB3 : K_GEMM32;

    // One launch group: m matrices factored together on one stream.
    struct Grp {
        V *Ab;
        int *ipb, *infob;
        const int *bidx;
        int m;
        char *xbuf;
        hipStream_t st;
    };
    // panel at column c for every member, in launches of as many members as
    // keep their clusters co-resident; members b0.. of a launch use exchange
    // buffers b0.. (the interchange kernel reads member b's permutation there)
    auto panel = [&](const Grp &G, int c, int pslot) {
        const int P = (n - c + RW - 1) / RW;
        const int per = std::max(1, std::min(G.m, pl.resident / P));
        const double mr = n - c;
        for (int b0 = 0; b0 < G.m; b0 += per) {
            const int m = std::min(per, G.m - b0);
            PanelArgs<T> pa;
            pa.A = G.bidx ? G.Ab : G.Ab + (size_t)b0 * strideA;
            pa.lda = lda; pa.strideA = strideA; pa.n = n; pa.k = c;
            pa.P = P; pa.slots = pl.slots; pa.pslot = pslot;
            pa.ipiv = G.bidx ? G.ipb : G.ipb + (size_t)b0 * strideP;
            pa.strideP = strideP;
            pa.info = G.bidx ? G.infob : G.infob + b0;
            pa.err = ctx->d_err;
            pa.xbuf = G.xbuf + (size_t)b0 * X.mat_bytes;
            pa.bidx = G.bidx ? G.bidx + b0 : nullptr;
            pa.tagp = ctx->d_tag; pa.toff = (uint32_t)c;
            pa.nmem = d_nmem;
            // per column j, (mr-j) scalings and (mr-j)(NB-j-1) complex multiply-adds
            prof_begin(ctx, kPanelClass, G.st);
            hipLaunchKernelGGL((panel_kernel<T, TPR>()), dim3(P, m), dim3(256), 0, G.st, pa);
            prof_end(ctx, kPanelClass, G.st, m * 8.0 * (mr * NB * NB / 2.0 - (double)NB * NB * NB / 6.0),
                     m * 2.0 * mr * NB * esz);
        }
    };
    // interchanges of the panel at c (permutation slot ps) in columns [l0, l1),
    // solve for [tr0, tr1) with (do_swap) or without them, interchanges in [sw0, n)
    auto swap = [&](const Grp &G, int c, int ps, int l0, int l1, int tr0, int tr1, int sw0, int do_swap) {
        SwapArgs sa;
        sa.n = n; sa.k = c; sa.slots = pl.slots; sa.pslot = ps; sa.do_swap = do_swap;
        sa.nmem = d_nmem;
        sa.c_l0 = l0; sa.c_l1 = l1;
        sa.c_tr0 = tr0; sa.c_tr1 = tr1;
        sa.c_sw0 = sw0;
        prof_begin(ctx, kSwapClass, G.st);
        launch_swap<T>(ctx, sa, G.Ab, lda, strideA, G.xbuf, G.bidx, G.m, G.st);
        prof_end(ctx, kSwapClass, G.st, G.m * 4.0 * NB * NB * std::max(0, tr1 - tr0), G.m * 4.0 * NB * n * esz);
    };
    auto gemm = [&](const Grp &G, int r0, int c0, int mrows, int ncols, int kk, int K) {
        if (mrows <= 0 || ncols <= 0) return;
        const GemmArgs g{r0, c0, mrows, ncols, kk, K, d_nmem};
        // C read and written, L and U read once; flops of the kernel's algorithm:
        // three real products per complex multiply-add (6 flops) for complex128
        // and complex64, four FP32-equivalent real products (8 flops, each taken
        // as three bf16 products) for split-BF16x3
        const double fpc = gk == 2 ? 8.0 : 6.0;
        prof_begin(ctx, kGemmClass, G.st);
        launch_gemm(gk, G.Ab, lda, strideA, g, G.m, G.bidx, G.st);
        prof_end(ctx, kGemmClass, G.st, G.m * fpc * mrows * ncols * K,
                 G.m * (2.0 * mrows * ncols + (double)(mrows + ncols) * K) * esz);
    };

    {
        Grp G;
        G.m = batch;
        G.Ab = A;
        G.ipb = ipiv;
        G.infob = d_info;
        G.bidx = d_bidx;
        G.xbuf = xbase;
        G.st = s;
        hipLaunchKernelGGL(k_tag_bump, dim3(1), dim3(64), 0, s, ctx->d_tag, (uint32_t)n);
        // Outer blocks of kSub panels: inside a block the panels are applied to
        // the block's own columns at once, while the columns to the right get
        // their interchanges at once and their update from the whole block in
        // one product with K = kSub * NB (rows of the later panels' solves are
        // updated first by a short product).
        for (int k = 0; k < n && !side; k += kSub * NB) {
            const int kend = (n - k < kSub * NB) ? n : k + kSub * NB;
            for (int c = k; c < kend; c += NB) {
                if (c > k) gemm(G, c, c, n - c, kend - c, c - NB, NB);
                panel(G, c, 0);
                if (c == k) {
                    swap(G, c, 0, 0, c, c + NB, n, n, 1);
                } else {
                    swap(G, c, 0, 0, c, c + NB, kend, kend, 1);
                    if (kend < n) {
                        gemm(G, c, kend, NB, n - kend, k, c - k);
                        swap(G, c, 0, 0, 0, kend, n, n, 0);
                    }
                }
            }
            gemm(G, kend, kend, n - kend, n - kend, k, kend - k);
        }
        // Look-ahead: a block's update goes to the next block's columns first; the
        // rest of it runs on the side stream while the next block's panels (which
        // leave most of the device idle) are factored inside their own columns.
        // Their interchanges and solves of the other columns wait for both.  Every
        // entry takes the same operations in the same order: the same bits.
        Grp H = G;
        H.st = side;
        bool pending = false;
        for (int k = 0; k < n && side; k += kSub * NB) {
            const int kend = std::min(n, k + kSub * NB), kend2 = std::min(n, kend + kSub * NB);
            for (int c = k; c < kend; c += NB) {
                if (c > k) gemm(G, c, c, n - c, kend - c, c - NB, NB);
                panel(G, c, (c - k) / NB);
                swap(G, c, (c - k) / NB, k, c, c + NB, kend, n, 1);
            }
            if (pending) WM_HIP_TRY(hipStreamWaitEvent(s, ctx->lu_ev[1], 0));
            pending = false;
            for (int c = k; c < kend; c += NB) {
                const int ps = (c - k) / NB;
                if (c == k) {
                    swap(G, c, ps, 0, k, kend, n, n, 1);
                } else {
                    swap(G, c, ps, 0, k, 0, 0, kend, 1);
                    if (kend < n) {
                        gemm(G, c, kend, NB, n - kend, k, c - k);
                        swap(G, c, ps, 0, 0, kend, n, n, 0);
                    }
                }
            }
            if (kend2 < n) {
                WM_HIP_TRY(hipEventRecord(ctx->lu_ev[0], s));
                WM_HIP_TRY(hipStreamWaitEvent(side, ctx->lu_ev[0], 0));
                gemm(H, kend, kend2, n - kend, n - kend2, k, kend - k);
                WM_HIP_TRY(hipEventRecord(ctx->lu_ev[1], side));
                pending = true;
            }
            gemm(G, kend, kend, n - kend, kend2 - kend, k, kend - k);
        }
        WM_HIP_TRY(hipGetLastError());
    }
    return WM_OK;
}

}  // namespace

int getrf_block(const wm_ctx *ctx, int prec, int n)
{
    const int dflt = n >= kSubLargeN ? kSubLarge : kSubDefault;
    if (prec < 0 || prec > 2) return dflt;
    const int sc = std::min(n / 1024, wm_ctx::kTuneSizes - 1);
    const int v = ctx->getrf_block[prec][sc];
    return v > 0 ? v : dflt;
}

int getrf_width(wm_ctx *ctx, int prec, int n)
{
    int bpc = 0;
    const bool f64 = prec == WM_PREC_F64;  // complex64 factors (FP32, BF16X3) share the FP32 panel
    if ((f64 ? occupancy_panel<double, kTprF64>(&bpc) : occupancy_panel<float, kTprF32>(&bpc)) != WM_OK || bpc <= 0) return 1;
    const int RW = 256 / (f64 ? kTprF64 : kTprF32);
    const int pmax = (n + RW - 1) / RW;
    return std::max(1, bpc * ctx->num_cu / std::max(1, ctx->panel_share) / pmax);
}

namespace {

// Enqueues a whole factorization (info reset, tag bumps, all launch chunks).
template <typename T, int TPR>
int getrf_enqueue(wm_ctx *ctx, const GetrfPlan &pl, int n, void *A, int lda, int64_t strideA, int *ipiv,
                  int64_t strideP, int batch, int *d_info, const int *d_bidx, hipStream_t s, int gk, int ks,
                  const int *d_nmem, hipStream_t side)
{
    if (!d_bidx) hipLaunchKernelGGL(k_zero_int, dim3((batch + 255) / 256), dim3(256), 0, s, d_info, batch);
    else hipLaunchKernelGGL(k_zero_idx, dim3((batch + 255) / 256), dim3(256), 0, s, d_info, d_bidx, batch);
    return getrf_impl<T, TPR>(ctx, pl, n, (typename CT<T>::V *)A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx,
                              s, gk, ks, d_nmem, side);
}

// Look-ahead stream of a factorization, or null for one that runs on one stream.
// The side stream pays once its updates are long enough against the launches and
// events it adds (1 x 4096: 14.1 -> 14.4 ms, 4 x 4096: 21.9 -> 21.6, 12 x 4096: 44.4 ->
// 43.8, 2 x 8192: 63.8 -> 61.4, 2 x 14336: 246 -> 236; split-BF16x3 12 x 8192: 117 ->
// 110 ms) and while the panels of the batch go in one launch, which leaves CUs
// idle; a batch of several such launches keeps the device busy by itself (16 x
// 8192: 347 -> 360 ms).  The profiler keeps every launch on one stream.
constexpr int64_t kSideMinEntries = (int64_t)1 << 26;
int getrf_side(wm_ctx *ctx, const GetrfPlan &pl, int n, int batch, int ks, hipStream_t *side)
{
    *side = nullptr;
    if (ctx->prof.on || batch > pl.per_launch || n <= 2 * ks * NB || (int64_t)n * n * batch < kSideMinEntries)
        return WM_OK;
    if (!ctx->lu_side) {  // events first, the stream last: lu_side set means all exist
        for (auto &e : ctx->lu_ev)
            if (!e) WM_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        WM_HIP_TRY(hipStreamCreateWithFlags(&ctx->lu_side, hipStreamNonBlocking));
    }
    *side = ctx->lu_side;
    return WM_OK;
}

// The contexts of one device, whose factorizations may run at the same time.
// A panel cluster's workgroups wait for each other, so every cluster that may be
// dispatched in part has to fit on the device beside the others': the lanes of a
// server share it by panel_share, contexts of several host threads by this gate.
// A factorization whose largest cluster does not fit beside those still running
// starts behind them (an event, no wait on the host); clusters of 64 rows per
// workgroup would otherwise fill the device at half the rows that those of 128
// did (four threads with one matrix of N = 14336 each: 896 of 768 workgroups).
// Counted per XCD, to which a launch deals its workgroups round-robin.
// One context alone pays two uncontended locks.
struct PanelGate {
    std::mutex mu;
    std::condition_variable cv;  // a context has finished enqueuing
    std::vector<wm_ctx *> live;
};
constexpr int kGateDevices = 64;
PanelGate g_gates[kGateDevices];

class PanelHold {
    static constexpr int kXcds = 8;
    wm_ctx *c_;
    hipStream_t s_;

    static int per_xcd(int workgroups) { return (workgroups + kXcds - 1) / kXcds; }

public:
    PanelHold(wm_ctx *c, hipStream_t s) : c_(c), s_(s) {}
    // device_total(int *): panel workgroups that the device holds
    template <typename F>
    int enter(int cluster, F device_total)
    {
        PanelGate &g = g_gates[c_->device];
        std::unique_lock<std::mutex> lk(g.mu);
        hipError_t e = hipSuccess;
        int total = 0;
        if (g.live.size() > 1) WM_TRY(device_total(&total));
        for (bool fits = total == 0; !fits;) {
            int sum = per_xcd(cluster);
            bool enqueuing = false;
            for (wm_ctx *o : g.live) {
                if (o == c_) continue;
                if (o->lu_phase == wm_ctx::LU_RECORDED && hipEventQuery(o->lu_done) == hipSuccess)
                    o->lu_phase = wm_ctx::LU_NONE;
                if (o->lu_phase == wm_ctx::LU_NONE) continue;
                sum += per_xcd(o->lu_cluster);
                enqueuing = enqueuing || o->lu_phase == wm_ctx::LU_ENQUEUING;
            }
            (void)hipGetLastError();  // an event that is not ready is no error
            fits = sum <= total / kXcds;
            if (!fits && enqueuing) {  // it has no event to wait for yet
                g.cv.wait(lk);
                continue;
            }
            if (!fits)
                for (wm_ctx *o : g.live)
                    if (o != c_ && o->lu_phase == wm_ctx::LU_RECORDED && e == hipSuccess)
                        e = hipStreamWaitEvent(s_, o->lu_done, 0);
            fits = true;
        }
        // the one before on this stream may still run
        if (c_->lu_phase == wm_ctx::LU_RECORDED && hipEventQuery(c_->lu_done) != hipSuccess) {
            (void)hipGetLastError();
            cluster = std::max(cluster, c_->lu_cluster);
        }
        c_->lu_phase = wm_ctx::LU_ENQUEUING;
        c_->lu_cluster = cluster;
        lk.unlock();
        WM_HIP_TRY(e);
        return WM_OK;
    }
    ~PanelHold()
    {
        PanelGate &g = g_gates[c_->device];
        std::lock_guard<std::mutex> lk(g.mu);
        if (c_->lu_phase != wm_ctx::LU_ENQUEUING) return;
        c_->lu_phase = wm_ctx::LU_NONE;
        if (g.live.size() > 1) {
            if ((c_->lu_done || hipEventCreateWithFlags(&c_->lu_done, hipEventDisableTiming) == hipSuccess) &&
                hipEventRecord(c_->lu_done, s_) == hipSuccess)
                c_->lu_phase = wm_ctx::LU_RECORDED;
            else
                (void)hipStreamSynchronize(s_);  // no event: finished before anyone else starts
        }
        g.cv.notify_all();
    }
};

template <typename T, int TPR>
int getrf_run(wm_ctx *ctx, int prec, int n, void *A, int lda, int64_t strideA, int *ipiv, int64_t strideP, int batch,
              int *d_info, const int *d_bidx, hipStream_t s, int gk, const int *d_nmem)
{
    const int ks = getrf_block(ctx, prec, n);
    GetrfPlan pl;
    if constexpr (!kTall<T, TPR>) {
        int resident = 0;
        WM_TRY((panel_resident<T, TPR>(ctx, &resident)));
        if ((n + 256 / TPR - 1) / (256 / TPR) > resident)
            return getrf_run<T, TPR / 2>(ctx, prec, n, A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx, s, gk,
                                         d_nmem);
    }
    WM_TRY((getrf_plan<T, TPR>(ctx, n, batch, &pl)));
    const uint64_t ntags = (uint64_t)n;
    WM_TRY(prepare_xbuf(ctx, pl.xbytes, ntags, s));
    hipStream_t side = nullptr;
    WM_TRY(getrf_side(ctx, pl, n, batch, ks, &side));
    PanelHold hold(ctx, s);
    WM_TRY(hold.enter(pl.pmax, [&](int *total) { return panel_total<T, TPR>(ctx, total); }));
    if (!ctx->use_graphs || ctx->prof.on) {
        WM_TRY((getrf_enqueue<T, TPR>(ctx, pl, n, A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx, s, gk, ks,
                                      d_nmem, side)));
    } else {
        // Replay a captured factorization of the same shape and buffers, or
        // capture one.  Its kernels read their tags from the device counter, so
        // every replay uses fresh tags.
        const GraphKey key{(int64_t)prec, (int64_t)n, (int64_t)lda, strideA, (int64_t)(intptr_t)A,
                           (int64_t)(intptr_t)ipiv, strideP, (int64_t)batch, (int64_t)(intptr_t)d_info,
                           (int64_t)(intptr_t)d_bidx, (int64_t)ks, (int64_t)(intptr_t)ctx->ws_lu.ptr,
                           (int64_t)(intptr_t)d_nmem};
        hipGraphExec_t exec = find_graph(ctx, key);
        if (!exec) {
            WM_HIP_TRY(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            const int rc = getrf_enqueue<T, TPR>(ctx, pl, n, A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx, s,
                                                 gk, ks, d_nmem, side);
            hipGraph_t graph = nullptr;
            const hipError_t ec = hipStreamEndCapture(s, &graph);
            if (rc != WM_OK) {
                if (graph) (void)hipGraphDestroy(graph);
                return rc;
            }
            WM_HIP_TRY(ec);
            const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            WM_HIP_TRY(ei);
            keep_graph(ctx, key, exec);
        }
        WM_HIP_TRY(hipGraphLaunch(exec, s));
    }
    ctx->panel_tag += ntags;
    return WM_OK;
}

}  // namespace

int panel_gate_join(wm_ctx *ctx)
{
    if (ctx->device < 0 || ctx->device >= kGateDevices) {
        set_error("device %d beyond %d", ctx->device, kGateDevices);
        return WM_ERR_ARG;
    }
    PanelGate &g = g_gates[ctx->device];
    std::unique_lock<std::mutex> lk(g.mu);
    // a context that was alone has recorded nothing behind its factorizations:
    // they end before it has company
    if (g.live.size() == 1) {
        g.cv.wait(lk, [&] { return g.live.size() != 1 || g.live[0]->lu_phase != wm_ctx::LU_ENQUEUING; });
        if (g.live.size() == 1) WM_HIP_TRY(hipStreamSynchronize(g.live[0]->stream));
    }
    g.live.push_back(ctx);
    return WM_OK;
}

void panel_gate_leave(wm_ctx *ctx)
{
    PanelGate &g = g_gates[ctx->device];
    std::lock_guard<std::mutex> lk(g.mu);
    g.live.erase(std::remove(g.live.begin(), g.live.end(), ctx), g.live.end());
    g.cv.notify_all();
}

// Destroys the captured factorizations.  A replay may still be running on the
// stream it was launched on (nothing waits for it before the exchange buffer
// grows or the cache fills), and HIP does not promise that an executable graph
// outlives its destruction while in flight, so the device is drained first.
void drop_graphs(wm_ctx *ctx)
{
    if (ctx->graphs.empty()) return;
    (void)hipSetDevice(ctx->device);
    (void)hipDeviceSynchronize();
    for (auto &kv : ctx->graphs) (void)hipGraphExecDestroy(kv.second);
    ctx->graphs.clear();
}

hipGraphExec_t find_graph(wm_ctx *ctx, const GraphKey &key)
{
    auto it = ctx->graphs.find(key);
    return it == ctx->graphs.end() ? nullptr : it->second;
}

void keep_graph(wm_ctx *ctx, const GraphKey &key, hipGraphExec_t exec)
{
    if (ctx->graphs.size() >= wm_ctx::kGraphCap) drop_graphs(ctx);
    ctx->graphs[key] = exec;
}

int getrf_batched(wm_ctx *ctx, int prec, int n, void *A, int lda, int64_t strideA, int *ipiv, int64_t strideP,
                  int batch, int *d_info, hipStream_t s, const int *d_bidx, const int *d_nmem)
{
    if (n <= 0 || n % NB != 0 || lda < n || batch <= 0 || !A || !ipiv || !d_info) {
        set_error("getrf: bad arguments (n=%d must be a positive multiple of %d, lda=%d, batch=%d)", n, NB, lda,
                  batch);
        return WM_ERR_ARG;
    }
    if (prec == WM_PREC_F64)
        return getrf_run<double, kTprF64>(ctx, prec, n, A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx, s, 8, d_nmem);
    if (prec == WM_PREC_F32)
        return getrf_run<float, kTprF32>(ctx, prec, n, A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx, s, 4,
                                         d_nmem);
    if (prec == WM_PREC_BF16X3)
        return getrf_run<float, kTprF32>(ctx, prec, n, A, lda, strideA, ipiv, strideP, batch, d_info, d_bidx, s, 2,
                                         d_nmem);
    set_error("getrf: precision %d not available", prec);
    return WM_ERR_ARG;
}

}  // namespace wm

// ---------------------------------------------------------------------------
// Internal test hooks (not part of include/wiremom.h).

// Caps the panel workgroups taken as co-resident (0 restores the occupancy
// query's count), so small factorizations split their panel launches as large
// ones do; drops captured factorizations, whose launch split it changes.
extern "C" int wmx_set_panel_resident(wm_ctx *ctx, int cap)
{
    if (!ctx || cap < 0) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    ctx->panel_resident_cap = cap;
    wm::drop_graphs(ctx);
    return WM_OK;
}

// Factors the members idx[0..count) of a batch through an index table (as the
// refinement levels do); info[m] receives member m's info word.
extern "C" int wmx_getrf_batched_idx(wm_ctx *ctx, int prec, int n, void *A, int lda, int64_t strideA, int *ipiv,
                                     int64_t strideP, int count, int *info, const int *idx)
{
    using namespace wm;
    if (!ctx || count <= 0 || !idx || !info) return WM_ERR_ARG;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    int nm = 0;
    for (int i = 0; i < count; ++i) nm = std::max(nm, idx[i] + 1);
    int *d = nullptr;
    WM_HIP_TRY(hipMalloc(&d, sizeof(int) * (size_t)(count + nm)));
    int rc = copy_h2d(d, idx, sizeof(int) * count, ctx->stream);
    if (rc == WM_OK) rc = getrf_batched(ctx, prec, n, A, lda, strideA, ipiv, strideP, count, d + count, ctx->stream, d);
    if (rc == WM_OK) rc = check_device_error(ctx, ctx->stream);
    std::vector<int> h(nm, 0);
    if (rc == WM_OK) rc = copy_d2h(h.data(), d + count, sizeof(int) * nm, ctx->stream);
    for (int i = 0; i < count && rc == WM_OK; ++i) info[i] = h[idx[i]];
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipFree(d);
    return rc;
}

// One update of the right-looking factorization on a device matrix (n x n, lda = n,
// complex128 for prec 0, complex64 else), without the factorization: C -= L U with
// C = A[k+NB.., k+NB..], L = A[k+NB.., k..k+NB), U = A[k..k+NB, k+NB..).
extern "C" int wmx_gemm_step(wm_ctx *ctx, int prec, int n, void *A, int k)
{
    using namespace wm;
    const int m2 = n - k - NB;
    if (m2 <= 0 || n % NB || k % NB) return WM_ERR_ARG;
    const GemmArgs g{k + NB, k + NB, m2, m2, k, NB, nullptr};
    launch_gemm(prec == WM_PREC_F64 ? 8 : prec == WM_PREC_BF16X3 ? 2 : 4, A, n, 0, g, 1, nullptr, ctx->stream);
    WM_HIP_TRY(hipStreamSynchronize(ctx->stream));
    return WM_OK;
}
