// Impedance-matrix fill for gfx950.
//
// Replaces the reference's CPU fill zmatrix()/wim() ("wersja referencyjna/
// Zmatrix.cpp":27-233) and its six-pass CUDA fill (zmatrix_gpu,
// "wersja referencyjna/Wire_MoM.cu":4052-4197; kernels at 520, 851, 1856, 2189,
// 3200, 3407).  One launch writes every entry of up to kMaxF frequency
// matrices exactly once:
//
//   Z[m,n] = j*eta0/(4 pi k) * sum_{h=obs half of m} ( k^2 * sum_g (l_g . l_h) V_hg  -+  sum_g +-S_hg / dl_g )
//
// where for source half g of basis n, V_hg / S_hg are the vector / scalar
// potential integrals (weights s/dl, (dl-s)/dl and 1) of exp(-jkR)/R taken
// with the reference's 2-point Gauss-Legendre rule, except on the self
// segment, where the singularity-extracted FP64 integrals (4-point rules on
// both halves plus the analytic log term, Zmatrix.cpp:279-323, 695-770) are
// precomputed per (basis, half, frequency) by k_self_terms.
//
// Mapping.  Every half is one segment, and a segment is shared by the bases at
// its two ends, so the kernel is evaluated once per pair (observation point,
// source segment) instead of once per pair of halves (four times as often):
//  * a wave owns a run of rows whose observation points are at most 64 distinct
//    ones (about 60 rows; wm_geom's tables): lane p evaluates point p, and the
//    rows' lanes gather the values of their two points through LDS (within the
//    wave: no barrier);
//  * it walks a run of source bases n (wave-uniform, so the records arrive
//    through scalar loads) and keeps the last segment's contribution as a first
//    half: along a wire the second half of basis n is the first half of n + 1.
// Measured at N = 8192, four frequencies: 968 -> 368 us per frequency (PEC ground
// 1748 -> 679 us); N = 511: 25 -> 7.5 us.  The launch is bound by the vector units (active
// in 84 % of the SIMD cycles at three waves per SIMD, 70 % with the complex64 copy;
// writing the matrix alone would take about 220 us): R, 1/R and the two nodes' weights are shared by the
// frequencies, and per frequency and pair a lane issues about 105 instructions.
// The four-term difference of scalar potentials is taken from values that are
// the same bits in every entry that uses a pair, scalar and vector parts summed
// apart, so the rounding errors of the potentials cancel around loops as the
// potentials do.  R and 1/R are shared by every frequency of the launch: the
// kernel e^{-jkR}/R is taken as (cos kR, -sin kR) * (1/R), 1/R from one
// reciprocal square root of R^2 per quadrature point and R = R^2 (1/R), where
// the reference takes a square root and divides ("wersja referencyjna/
// Zmatrix.cpp":679-688); the results differ from its by about an ulp.
// cos kR and sin kR come from sincos_phase (wm_sincos.h: Cody-Waite reduction
// and minimax polynomials, within about 1.5 ulp of the exact values for kR up
// to 100 and 2.5 ulp up to its limit), which needs a fraction of the
// operations and registers of a general-purpose sincos.
//
// PEC ground (ienv 2, "wersja referencyjna/Zmatrix.cpp":94-145, 174-224): every
// source half is followed by its image in z = 0 (coordinates scaled by the
// environment signs, weight sgnenv), which doubles the kernel evaluations.
#include <algorithm>

#include "wm_internal.h"
#include "wm_sincos.h"

namespace wm {

namespace {

constexpr int kMaxF = 4;          // frequencies per launch (with or without the image terms)
constexpr int kWaves = 4;         // waves per block
constexpr int kMinCols = 4, kMaxCols = 32;  // source bases per wave
constexpr double kPi = 3.14159265358979323846;
constexpr double kGL2 = 0.288675134594812882;  // 2-point node offset / length
constexpr double kGL4c1 = 0.43056815579702629, kGL4w1 = 0.17392742256872693;
constexpr double kGL4c2 = 0.16999052179242813, kGL4w2 = 0.32607257743127307;

typedef double d2v __attribute__((ext_vector_type(2)));

struct FreqArgs {
    double ka[kMaxF];
    double ka2[kMaxF];  // 2 k^2
    double q[kMaxF];    // eta0 / (8 pi k)
    int64_t zo[kMaxF];  // offset of each frequency's matrix from Z (elements)
};

// Complete elliptic K from the Abramowitz & Stegun 17.3.34 polynomial in
// m1 = 1 - bet^2 with the reference's truncation thresholds (Zmatrix.cpp:731-770).
__device__ double elliptic_k_as(double bet)
{
    const double m1 = 1.0 - bet * bet;
    double a = 1.38629436112 + 0.09666344259 * m1;
    double b = 0.5 + 0.12498593597 * m1;
    double m12 = 0.0, m13 = 0.0;
    if (m1 >= 1.0e-18) { m12 = m1 * m1; a += 0.03590092383 * m12; b += 0.06880248576 * m12; }
    if (m1 >= 1.0e-12) { m13 = m12 * m1; a += 0.03742563713 * m13; b += 0.03328355346 * m13; }
    if (m1 >= 1.0e-9) { const double m14 = m13 * m1; a += 0.01451196212 * m14; b += 0.00441787012 * m14; }
    return a - b * log(m1);
}

// Singularity-extracted self kernel at offset s along a segment of length dl
// and radius an (Zmatrix.cpp:695-728, before the ifun weight).
__device__ double2 self_kernel(double s, double ka, double dl, double an)
{
    const double r = 0.5 * dl - s;
    const double rr = sqrt(an * an + r * r);
    double sn, cn;
    sincos(ka * rr, &sn, &cn);
    const double c1r = (cn - 1.0) / rr, c1i = (-sn) / rr;
    const double bet = (an + an) / sqrt(4.0 * an * an + r * r);
    const double bnd2 = (bet * elliptic_k_as(bet) + log(fabs(r / (8.0 * an)))) / (kPi * an);
    return make_double2(c1r + bnd2, c1i);
}

// Integrals over the self segment (Zmatrix.cpp:279-323): 4-point rules on both
// halves of the segment plus the analytic log term.
// self[(f*ld + n)*4 + 2*g + {0: vector, 1: scalar}] for source half g of n.
// Eight lanes per (n, g), one quadrature node each, shared by the vector and
// the scalar integral, their sums in fixed order (one lane per (n, g) took all
// 16 kernel evaluations and F frequencies in turn: 20 us per frequency at any
// size, most of a small fill).
__global__ __launch_bounds__(256) void k_self_terms(const double *__restrict__ src, int npls, int ld, FreqArgs fa,
                                                    double2 *__restrict__ self)
{
    const int t = blockIdx.x * 256 + threadIdx.x, f = blockIdx.y;
    const int node = t & 7, n = t >> 4, g = (t >> 3) & 1;
    if (n >= ld) return;  // uniform over the eight lanes
    double2 v = make_double2(0.0, 0.0), s = v;
    if (n < npls) {
        const double dl = src[(size_t)n * 16 + g * 8 + 6];
        const double an = src[(size_t)n * 16 + g * 8 + 7];
        const double dlh = 0.5 * dl;
        const double xl = node & 4 ? dlh : 0.0, xu = node & 4 ? dl : dlh;
        const double b = xu - xl, c = (node & 2 ? kGL4c2 : kGL4c1) * b, w = node & 2 ? kGL4w2 : kGL4w1;
        const double x = 0.5 * (xl + xu) + (node & 1 ? -c : c);
        s = self_kernel(x, fa.ka[f], dl, an);
        const double wt = g == 0 ? x / dl : (dl - x) / dl;
        v = make_double2(s.x * wt, s.y * wt);
        auto total = [&](double y) {  // ((+ node) + (- node)) w, the two pairs, b, the two halves
            y = (y + __shfl_xor(y, 1)) * w;
            y = (y + __shfl_xor(y, 2)) * b;
            return y + __shfl_xor(y, 4);
        };
        const double res = dl * (1.0 + log(16.0 * an / dl)) / (kPi * an);
        v = make_double2(total(v.x) + 0.5 * res, total(v.y));
        s = make_double2(total(s.x) + res, total(s.y));
    }
    if (node == 0) {
        self[((size_t)f * ld + n) * 4 + 2 * g] = v;
        self[((size_t)f * ld + n) * 4 + 2 * g + 1] = s;
    }
}

// The geometry's device tables (wm_geom) and the launch's share of the columns.
struct FillArgs {
    const double *obs;    // 12 arrays of ld doubles: rc1, lm1, rc2, lm2 per row
    const double *pts;    // per wave of rows 3 x 64 doubles: observation points x, y, z
    const int *pkey;      // and 64 ints: their segment keys
    const int *wrow;      // first row of each wave
    const int *slots;     // per row: its two points' lanes, first | second << 8
    int nwaves, npls, ld, cols;
    const double *src;    // source records
    const int *skey;      // 4 ints per basis: keys of its halves, 1 if its first half is not the second of n - 1, 0
    // PEC ground (IMG): after each source half its image is taken with the same
    // rule -- the self rule on the image of the observation segment itself when
    // that segment lies in the ground plane -- and added with weight sgnenv
    // ("wersja referencyjna/Zmatrix.cpp":86-151, 167-231)
    const double *img;    // image records, as src
    const int *ikey;      // image self keys, 2 per basis
    double sgnenv;
};

template <int F, bool kW32, bool IMG>
__global__ __launch_bounds__(64 * kWaves) void k_fill(FillArgs a, const double2 *__restrict__ self, FreqArgs fa,
                                                      double2 *__restrict__ Z, float2 *__restrict__ Z32,
                                                      int64_t strideZ32)
{
    // Every rounding is spelled out (fma where fused), so an entry does not
    // depend on how many frequencies share the launch (F) or on the columns per
    // wave: the compiler may not contract products differently per instantiation.
#pragma clang fp contract(off)
    constexpr int NP = IMG ? 2 : 1;
    constexpr double kW1 = 0.5 + kGL2, kW0 = 0.5 - kGL2;  // weight s/dl at the two nodes
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wv = blockIdx.x * kWaves + wave;
    if (wv >= a.nwaves) return;
    // values of this wave's points for one frequency: VA, VB and 2 P, re and im
    // each; two buffers, so a frequency's gather overlaps the next one's kernel
    __shared__ double s_ex[kWaves][2][6][64];

    const int row0 = a.wrow[wv], row1 = a.wrow[wv + 1];
    const int m = row0 + lane;
    const bool isrow = m < row1;
    const int mr = isrow ? m : row0;
    double lm[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int d = 0; d < 3; ++d) lm[h][d] = a.obs[(size_t)(6 * h + 3 + d) * a.ld + mr];
    const int sl = a.slots[mr], sl0 = sl & 63, sl1 = (sl >> 8) & 63;
    double rc[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) rc[d] = a.pts[((size_t)wv * 3 + d) * 64 + lane];
    const int pkey = a.pkey[(size_t)wv * 64 + lane];

    // the polynomials' coefficients in vector registers: as scalar constants
    // they and the arguments exceed the scalar registers, and each use of a
    // spilled one costs a lane read
    SinCosConsts sk;
#pragma unroll
    for (int i = 0; i < 7; ++i) asm("" : "+v"(sk.s[i]));
#pragma unroll
    for (int i = 0; i < 6; ++i) asm("" : "+v"(sk.c[i]));

    // the open first half of the next column: sum_h (l_h . dc) V_A(h) and 2 P(1) - 2 P(0)
    double2 vp[F], dp[F];
#pragma unroll
    for (int f = 0; f < F; ++f) vp[f] = dp[f] = make_double2(0.0, 0.0);

    const int n0 = blockIdx.y * a.cols, n1 = min(a.ld, n0 + a.cols);
    for (int n = n0; n < n1; ++n) {
        if (n >= a.npls) {  // padding: the identity
            if (isrow) {
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    const size_t idx = (size_t)m + (size_t)n * a.ld;
                    const double one = m == n ? 1.0 : 0.0;
                    Z[fa.zo[f] + idx] = make_double2(one, 0.0);
                    if (kW32) Z32[f * strideZ32 + idx] = make_float2((float)one, 0.f);
                }
            }
            continue;
        }
        for (int g = n == n0 || a.skey[4 * n + 2] ? 0 : 1; g < 2; ++g) {
            // lane = point: distances to the segment's (and its image's) two nodes
            // (R, 1/R and 1/R times the nodes' weights of the two vector integrals)
            double R[NP][2], rR[NP][2], wa[NP][2], wb[NP][2], t[NP][2];
            bool own[NP];
            double dl[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const double *sr = (p ? a.img : a.src) + (size_t)n * 16 + 8 * g;
                own[p] = pkey == (p ? a.ikey[2 * n + g] : a.skey[4 * n + g]);
                const double dcx = sr[3], dcy = sr[4], dcz = sr[5], an = sr[7];
                dl[p] = sr[6];
                const double half = 0.5 * dl[p], off = kGL2 * dl[p];
                const double hw1 = half * kW1, hw0 = half * kW0;
                const double bx = rc[0] - sr[0], by = rc[1] - sr[1], bz = rc[2] - sr[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const double s = q == 0 ? half + off : half - off;
                    const double dx = fma(-s, dcx, bx), dy = fma(-s, dcy, by), dz = fma(-s, dcz, bz);
                    const double R2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, an * an)));
                    rR[p][q] = rsqrt(R2);
                    R[p][q] = R2 * rR[p][q];
                    wa[p][q] = (q == 0 ? hw1 : hw0) * rR[p][q];
                    wb[p][q] = (q == 0 ? hw0 : hw1) * rR[p][q];
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    t[p][h] = fma(dcz, lm[h][2], fma(dcy, lm[h][1], dcx * lm[h][0]));
                    if (p) t[p][h] *= a.sgnenv;
                }
            }
#pragma unroll
            for (int f = 0; f < F; ++f) {
                double2 va = make_double2(0.0, 0.0), vb = va, d = va;
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    double x[6];
                    {
                        double s1, c1, s0, c0;
                        sincos_phase(fa.ka[f] * R[p][0], s1, c1, sk);
                        sincos_phase(fa.ka[f] * R[p][1], s0, c0, sk);
                        x[0] = fma(wa[p][0], c1, wa[p][1] * c0);
                        x[1] = fma(-wa[p][0], s1, -(wa[p][1] * s0));
                        x[2] = fma(wb[p][0], c1, wb[p][1] * c0);
                        x[3] = fma(-wb[p][0], s1, -(wb[p][1] * s0));
                        x[4] = fma(rR[p][0], c1, rR[p][1] * c0);
                        x[5] = fma(-rR[p][0], s1, -(rR[p][1] * s0));
                    }
                    if (own[p]) {
                        // the segment itself: as second half of n it is the first of n + 1
                        const double2 *e = self + ((size_t)f * a.ld + n) * 4;
                        const double2 ea = g == 0 ? e[0] : e[n + 1 < a.npls ? 4 : 0], eb = e[2], es = e[2 * g + 1];
                        x[0] = ea.x; x[1] = ea.y;
                        x[2] = eb.x; x[3] = eb.y;
                        x[4] = 2.0 * es.x / dl[p];
                        x[5] = 2.0 * es.y / dl[p];
                    }
                    double(*ex)[64] = s_ex[wave][(f * NP + p) & 1];
#pragma unroll
                    for (int i = 0; i < 6; ++i) ex[i][lane] = x[i];
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    // lane = row: its two points' values
                    va.x = fma(ex[0][sl1], t[p][1], fma(ex[0][sl0], t[p][0], va.x));
                    va.y = fma(ex[1][sl1], t[p][1], fma(ex[1][sl0], t[p][0], va.y));
                    vb.x = fma(ex[2][sl1], t[p][1], fma(ex[2][sl0], t[p][0], vb.x));
                    vb.y = fma(ex[3][sl1], t[p][1], fma(ex[3][sl0], t[p][0], vb.y));
                    const double pr = ex[4][sl1] - ex[4][sl0], pi = ex[5][sl1] - ex[5][sl0];
                    d.x = p ? fma(a.sgnenv, pr, d.x) : pr;
                    d.y = p ? fma(a.sgnenv, pi, d.y) : pi;
                    __builtin_amdgcn_wave_barrier();
                }
                if (g == 1) {
                    // 2 k^2 (vector part) + 2 (scalar part of the first half - the second's)
                    const double ar = fma(vp[f].x + vb.x, fa.ka2[f], dp[f].x - d.x);
                    const double ai = fma(vp[f].y + vb.y, fa.ka2[f], dp[f].y - d.y);
                    const bool inside = m < a.npls;  // rows beyond: the identity
                    const double2 z = inside ? make_double2(-fa.q[f] * ai, fa.q[f] * ar) : make_double2(0.0, 0.0);
                    const size_t idx = (size_t)m + (size_t)n * a.ld;
                    if (isrow) {
                        // non-temporal: written once, read by a later kernel
                        __builtin_nontemporal_store(d2v{z.x, z.y}, (d2v *)&Z[fa.zo[f] + idx]);
                        if (kW32) Z32[f * strideZ32 + idx] = make_float2((float)z.x, (float)z.y);
                    }
                }
                vp[f] = va;
                dp[f] = d;
            }
        }
    }
}

template <int F>
void launch_fill(dim3 grid, hipStream_t s, const FillArgs &a, const double2 *self, const FreqArgs &fa, double2 *Z,
                 float2 *Z32, int64_t sZ32)
{
    const dim3 blk(64 * kWaves);
    if (a.img) {
        if (Z32) hipLaunchKernelGGL((k_fill<F, true, true>), grid, blk, 0, s, a, self, fa, Z, Z32, sZ32);
        else hipLaunchKernelGGL((k_fill<F, false, true>), grid, blk, 0, s, a, self, fa, Z, Z32, sZ32);
    } else {
        if (Z32) hipLaunchKernelGGL((k_fill<F, true, false>), grid, blk, 0, s, a, self, fa, Z, Z32, sZ32);
        else hipLaunchKernelGGL((k_fill<F, false, false>), grid, blk, 0, s, a, self, fa, Z, Z32, sZ32);
    }
}

}  // namespace

int fill_launch(wm_ctx *ctx, const wm_geom *g, int nf, const double *ka, void *Z, int64_t strideZ,
                void *Z32, int64_t strideZ32, hipStream_t s, DevBuf *self_ws, const int *slots)
{
    if (!g || nf <= 0 || !ka || !Z || (slots && Z32)) {
        set_error("fill: bad arguments");
        return WM_ERR_ARG;
    }
    const int ld = g->ld;
    // self-term workspace: kMaxF * ld * 4 complex128
    const size_t self_bytes = (size_t)kMaxF * ld * 4 * sizeof(double2);
    DevBuf &ws = self_ws ? *self_ws : ctx->ws_fill;
    WM_TRY(ws.ensure(self_bytes));
    double2 *self = (double2 *)ws.ptr;
    // Columns per wave: the first costs one more segment, so as many as leave
    // about 8 waves per SIMD of the device
    FillArgs fl;
    fl.obs = g->d_obs; fl.pts = g->d_pts; fl.pkey = g->d_pkey; fl.wrow = g->d_wrow; fl.slots = g->d_slots;
    fl.nwaves = g->nwaves; fl.npls = g->npls; fl.ld = ld;
    fl.cols = std::max(kMinCols, std::min(kMaxCols, (int)((int64_t)g->nwaves * ld / (32 * ctx->num_cu))));
    fl.src = g->d_src; fl.skey = g->d_src_key; fl.img = g->d_img; fl.ikey = g->d_img_key; fl.sgnenv = g->sgnenv;
    const dim3 grid((g->nwaves + kWaves - 1) / kWaves, (ld + fl.cols - 1) / fl.cols);
    // the phases k R stay inside the range of the fill's argument reduction
    // (R is at most the structure's diameter, images included, plus a radius)
    for (int f = 0; f < nf; ++f)
        if (!(ka[f] > 0.0) || ka[f] * (2.0 * g->diam + 1.0) >= kSinCosMax) {
            set_error("fill: wavenumber %g on a structure of diameter %g m is outside the fill's phase range", ka[f],
                      g->diam);
            return WM_ERR_ARG;
        }
    // frequencies per launch: the tuned setting for the environment and size, else kMaxF
    const int tuned = ctx->fill_freqs[g->ienv == 2 ? 1 : 0][std::min(ld / 1024, wm_ctx::kTuneSizes - 1)];
    const int fmax = tuned >= 1 && tuned <= kMaxF ? tuned : kMaxF;
    for (int f0 = 0; f0 < nf; f0 += fmax) {
        const int F = (nf - f0 < fmax) ? nf - f0 : fmax;
        FreqArgs fa;
        for (int f = 0; f < kMaxF; ++f) {
            const double k = ka[f0 + (f < F ? f : 0)];
            fa.ka[f] = k;
            fa.ka2[f] = 2.0 * k * k;
            fa.q[f] = 0.5 * (120.0 * kPi) / (4.0 * kPi * k);
            fa.zo[f] = (int64_t)(slots ? slots[f0 + (f < F ? f : 0)] : f0 + f) * strideZ;
        }
        hipLaunchKernelGGL(k_self_terms, dim3((16 * ld + 255) / 256, F), dim3(256), 0, s, g->d_src, g->npls, ld, fa, self);
        double2 *Zf = (double2 *)Z;  // each frequency's matrix at fa.zo[f]
        float2 *Z32f = Z32 ? (float2 *)Z32 + (size_t)f0 * strideZ32 : nullptr;
        // algorithmic count per frequency: 220 N^2 FP64 operations (440 N^2 with
        // the image terms of the PEC ground), 16 N^2 bytes written
        const double nn = (double)g->npls * g->npls;
        const double ops = g->ienv == 2 ? 440.0 : 220.0;
        prof_begin(ctx, K_FILL, s);
        switch (F) {
            case 1: launch_fill<1>(grid, s, fl, self, fa, Zf, Z32f, strideZ32); break;
            case 2: launch_fill<2>(grid, s, fl, self, fa, Zf, Z32f, strideZ32); break;
            case 3: launch_fill<3>(grid, s, fl, self, fa, Zf, Z32f, strideZ32); break;
            default: launch_fill<4>(grid, s, fl, self, fa, Zf, Z32f, strideZ32); break;
        }
        prof_end(ctx, K_FILL, s, ops * nn * F, (Z32 ? 24.0 : 16.0) * nn * F);
        WM_HIP_TRY(hipGetLastError());
    }
    return WM_OK;
}

}  // namespace wm
