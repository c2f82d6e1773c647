// Device-side complex helpers and the bounded cross-workgroup wait.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace wm {

template <typename T> struct CT;
template <> struct CT<double> { using V = double2; };
template <> struct CT<float> { using V = float2; };

// Spin limit for device-side waits: with the s_sleep below this is well
// over a second, far above any legitimate wait, and every waiting wave
// leaves once any wave has recorded a timeout in the error word.
constexpr long kSpinLimit = 1L << 24;

// Tagged 8-byte packets {32-bit tag, 32-bit payload} for data handed between
// workgroups of one grid: a reader polls a packet until its tag matches, so
// neither a counter nor a release/acquire fence (an L2 write-back and
// invalidate on gfx950) is needed.  8-byte loads and stores are single-copy
// atomic; agent-scope relaxed atomics reach the device coherence point.
__device__ inline void put_pkt(uint64_t *p, uint32_t tag, uint32_t v)
{
    __hip_atomic_store(p, ((uint64_t)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline uint64_t ld_pkt(const uint64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Bounded-wait bookkeeping for a polling lane: true if the lane must stop
// (the error word is set, or this lane ran out of spins and set it).
__device__ inline bool spin_give_up(long &it, int *err)
{
    if ((++it & 255) == 0) {
        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
        if (it > kSpinLimit) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return true;
        }
    }
    __builtin_amdgcn_s_sleep(1);
    return false;
}

// Reciprocal of a complex number, conj(z) / |z|^2 on z scaled by a power of two
// to a largest part in [1/2, 1): |z|^2 and its rounding error in two words, one
// hardware reciprocal refined by Newton steps, its remainder and the products'
// rounding errors folded into one last addition per part: within 0.51 ulp of
// the exact value (Smith's algorithm, three chained divisions: 1.4 ulp) in
// about a quarter of the dependent steps.  Zero and non-finite numbers take
// Smith's (1962) path.
__device__ inline double2 crecip(double re, double im)
{
    const double big = fmax(fabs(re), fabs(im));
    if (big > 0.0 && big < __builtin_inf() && re == re && im == im) {
        const int e = -__builtin_amdgcn_frexp_exp(big);
        const double a = __builtin_amdgcn_ldexp(re, e), b = __builtin_amdgcn_ldexp(im, e);
        const double aa = a * a, bb = b * b, d = aa + bb;
        const double lo = fmin(aa, bb) - (d - fmax(aa, bb));
        const double de = lo + (__builtin_fma(a, a, -aa) + __builtin_fma(b, b, -bb));
        double r = __builtin_amdgcn_rcp(d);
        r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
        r = __builtin_fma(r, __builtin_fma(-de, r, __builtin_fma(-d, r, 1.0)), r);
        const double q = __builtin_fma(-de, r, __builtin_fma(-d, r, 1.0));
        const double x = a * r, y = -b * r;
        return make_double2(__builtin_amdgcn_ldexp(x + __builtin_fma(x, q, __builtin_fma(a, r, -x)), e),
                            __builtin_amdgcn_ldexp(y + __builtin_fma(y, q, __builtin_fma(-b, r, -y)), e));
    }
    if (fabs(re) >= fabs(im)) {
        const double t = im / re, d = re + im * t;
        return make_double2(1.0 / d, -t / d);
    }
    const double t = re / im, d = im + re * t;
    return make_double2(t / d, -1.0 / d);
}

}  // namespace wm
