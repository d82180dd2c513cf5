// Donor errors of the K4 encoder from order-free sums, with a certificate.
//
// The reference's donor error of a channel is a float,
//     err = fl(fl(var) + fl(fl(fl(mean) - smean)^2)),
// with var and mean from a sequential fp64 Welford pass over the tokens
// (codec.py:207-210).  Only the order of these errors matters: the `count`
// least ones among the channels that are not sources form the donor pool.  A
// Welford pass is one dependent chain per channel, so the encoders take var
// and mean from fp64 sums of x and x^2 instead, which any number of lanes may
// share, and bound how far the chain's values can lie from them: `lo` and `hi`
// enclose the reference's float.  With the pool chosen by `lo`, the choice is
// the reference's whenever every pool member's `hi` key orders before every
// other candidate's `lo` key (iq_pool_certain); otherwise the row runs the
// Welford chains and selects again.
//
// The bound, u = 2^-53, A = the channel's largest magnitude, n tokens.  Every
// x is a float, so x^2 is exact in fp64.
//   mean   a chain step rounds by at most u (|mean| + 3 |delta| / k) with
//          |delta| <= 2 A, and step j's error reaches the end scaled by j / n:
//          at most (n / 2 + 7) u A in all; S1 / n adds at most (n + 1) u A.
//          E = (2 n + 32) u A encloses both.
//   var    delta and x - mean each carry a mean error below E' = (n + 8) u A,
//          so a term of the chain's sum is off by at most 4 A E', and its own
//          roundings and the sum's add (n + 3) u of a term of at most 4 A^2:
//          8 (n + 8) u A^2 after the division by n.  S2 / n - (S1 / n)^2 is
//          off by at most 4 (n + 16) u A^2.  H = 16 (n + 16) u A^2 encloses
//          both with a quarter to spare.
// A channel of zeros has E = H = 0: its error is exactly zero.  So is the error
// of a channel whose tokens all hold one value v (`same`): the chain's mean is v
// from its first step on, its sum stays zero, and err = fl(fl(v - smean)^2).
// Without that a block of equal tokens (padding, a run of one token) left every
// pool uncertain: relative to a variance of zero the bound is not small.
//
// Plain arithmetic, every operation rounded by itself (-ffp-contract=off), so
// that it compiles for the host too (tests/test_k4_rows.py).
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define IQ_HD __host__ __device__ __forceinline__
#else
#define IQ_HD static inline
#endif

struct IqErrRange {
    float lo, hi;
};

// Whether all of n <= 256 values of a 16-bit type are equal, from their sums.
// A value other than the largest in magnitude differs from it by at least
// 2^-11 A, so a channel that is not constant has a variance of at least
// 2^-22 A^2 / (2 n) >= 2^-31 A^2; the computed one is within
// 4 (n + 16) u A^2 < 2^-42 A^2 of the true one, and H < 2^-40 A^2.
IQ_HD bool iq_same16(double s1, double s2, float amax, int64_t n)
{
    const double inv = 1.0 / (double)n, A = (double)amax, mean = s1 * inv;
    return __builtin_fma(-mean, mean, s2 * inv) <= A * A * ((double)(n + 16) * 0x1p-49);
}

IQ_HD IqErrRange iq_err_range(double s1, double s2, float amax, float smean, int64_t n, bool same)
{
    if (same) {
        const float d = __builtin_copysignf(amax, (float)s1) - smean, q = d * d;
        return IqErrRange{q, q};
    }
    const double inv = 1.0 / (double)n, A = (double)amax;
    const double mean = s1 * inv;
    const double var = __builtin_fma(-mean, mean, s2 * inv);
    const double E = A * ((double)(2 * n + 32) * 0x1p-53);
    const double H = A * A * ((double)(n + 16) * 0x1p-49);
    const float vlo = (float)__builtin_fmax(var - H, 0.0), vhi = (float)__builtin_fmax(var + H, 0.0);
    const float da = (float)(mean - E) - smean, db = (float)(mean + E) - smean;
    // rounding is monotone: diff lies in [da, db], its square between these
    const float qa = da * da, qb = db * db;
    const float qlo = (da < 0.0f && db > 0.0f) ? 0.0f : __builtin_fminf(qa, qb), qhi = __builtin_fmaxf(qa, qb);
    IqErrRange r;
    r.lo = vlo + qlo;
    r.hi = vhi + qhi;
    return r;
}

// Errors in the order of the selection: ascending, ties to the lower channel.
IQ_HD uint64_t iq_err_key(float err, int c)
{
    uint32_t bits;
    __builtin_memcpy(&bits, &err, 4);
    return ((uint64_t)bits << 10) | (uint64_t)c;
}
