// Exact modular products in double precision for primes below 2^51 (device).
// fp_mulmod(a, w) with integers |a w| <= 2^53 q:
//   h = a w (rounded), e = fma(a, w, -h) = a w - h exactly,
//   Q = rint(h / q), off the quotient by at most 1/2 + 3 2^-53 |a w / q|,
//   r = fma(-Q, q, h) + e = a w - Q q,
// every intermediate an integer below 2^53, so r is exact: |r| <= 1.25 q for
// |a|, |w| <= q, and |r| <= q/2 + 1.5 2^-53 q |a| for centred |w| <= q/2.
// fp_reduce(z) = z - rint(z / q) q maps an integer |z| < 2^53 to a
// representative of magnitude at most q/2 (1 + eps).  Files using these are
// compiled without floating-point contraction.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nx {

constexpr uint64_t kFpPrime = 1ull << 51;  // primes below this take the double-precision forms

// p[i] of a table that no kernel writes, at an index that is the same for the
// whole wave: a scalar load.  Through an ordinary pointer the compiler has to
// assume that the kernel's own stores may reach the table, and takes a vector
// load, which waits for them.
template <class T>
__device__ __forceinline__ T table_at(const T *p, uint64_t i)
{
    typedef const __attribute__((address_space(4))) T *Constant;
    return ((Constant)(uintptr_t)p)[i];
}

// x < 2^52 as a double: two instructions (the compiler's conversion takes four)
__device__ __forceinline__ double fp_from(uint64_t x)
{
    return __longlong_as_double((long long)(x | 0x4330000000000000ull)) - 0x1p52;
}

// an integer 0 <= x < 2^52 as a word: two instructions instead of six
__device__ __forceinline__ uint64_t fp_to(double x)
{
    return (uint64_t)__double_as_longlong(x + 0x1p52) & 0x000fffffffffffffull;
}

__device__ __forceinline__ double fp_mulmod(double a, double w, double q, double qinv)
{
    const double h = a * w;
    const double e = __builtin_fma(a, w, -h);
    const double Q = __builtin_rint(h * qinv);
    return __builtin_fma(-Q, q, h) + e;
}

__device__ __forceinline__ double fp_reduce(double z, double q, double qinv)
{
    return __builtin_fma(-__builtin_rint(z * qinv), q, z);
}

// fp_reduce, then mapped to [0, q) as an integer
__device__ __forceinline__ uint64_t fp_final(double z, double q, double qinv)
{
    z = fp_reduce(z, q, qinv);
    return fp_to(z < 0 ? z + q : z);
}

// Sums of products with one division at the end.  S = sum a_i b_i is kept as
// H + L: the accumulator starts at M = 1.5 2^(52 + s), so every fma rounds to
// a multiple of 2^s while the sum of products stays below 2^(51 + s) in
// magnitude; the step it takes is exact (d = new - old) and what it left out,
// lo = a b - d with |lo| <= 2^(s - 1), is exact too and collects in L.  Four
// instructions a term, against eight and a half for fp_mulmod, the addition
// and a reduction every second term.
struct FpSum {
    double h, l;
    __device__ __forceinline__ void start(double M)
    {
        h = M;
        l = 0.0;
    }
    __device__ __forceinline__ void mac(double a, double b)
    {
        const double n = __builtin_fma(a, b, h);
        l += __builtin_fma(a, b, -(n - h));
        h = n;
    }
    // S mod q, |r| <= q/2 (1 + eps), for |S| / q <= 2^53 and |L| <= 2^53: the
    // quotient of H is within 2.5 of H / q, so r = H - Q q and r + L' (L'
    // reduced) stay below 2^53
    __device__ __forceinline__ double value(double M, double q, double qinv) const
    {
        const double H = h - M;
        const double r = __builtin_fma(-__builtin_rint(H * qinv), q, H);
        return fp_reduce(r + fp_reduce(l, q, qinv), q, qinv);
    }
};

// Inner products sum t_j k_j with |t| <= q/2 (1 + eps) and 0 <= k < q < 2^b:
// M and the number of terms T between two folds (value(), restarted with the
// folded sum in L).  Needs T 2^(2b - 1) <= 2^(51 + s) (range of the
// accumulator), T 2^(s - 1) + 2^(b - 1) <= 2^53 (L exact) and T 2^b <= 2^53
// (the quotient exact):
//   q < 2^47: s = 47, T = 32;  q < 2^50: s = 51, T = 7;  q < 2^51: s = 52, T = 3.
__device__ __forceinline__ double fp_inner_magic(uint64_t q)
{
    return q < (1ull << 47) ? 0x1.8p99 : (q < (1ull << 50) ? 0x1.8p103 : 0x1.8p104);
}
__device__ __forceinline__ uint32_t fp_inner_terms(uint64_t q)
{
    return q < (1ull << 47) ? 32u : (q < (1ull << 50) ? 7u : 3u);
}

// The same for |t| <= 2^50 and q < 2^47 (values a lazy transform left): T 2^97
// <= 2^(51 + s), T 2^(s - 1) + 2^46 <= 2^53 and T 2^50 <= 2^53 with s = 49, T = 8.
constexpr double kFpLazyMagic = 0x1.8p101;
constexpr uint32_t kFpLazyTerms = 8;

}  // namespace nx
