// Sequential FP64 sums out of order: the pieces of an exact parallel
// evaluation of s = (((s + v0) + v1) + ...), rounded after every addition, as
// the reference's tree takes its means (src/fmm.c:184-196).  Shared by the
// tree kernels and the host, where the rule is tested against the plain loop.
//
// While the running sum stays inside one binade [2^e, 2^(e+1)) every addition
// rounds to a multiple of the same unit u = 2^(e-52): s is an integer number S of
// units, and S + v / u rounds to S + rint(v / u) whatever S is, unless v / u lies
// exactly halfway between two integers.  A halfway case rounds to the even
// neighbour, S + floor(v / u) or one more, and leaves an even S; so its
// round-up bit is the parity of the integers added since the last halfway case
// (of S and those integers for the first one).  A batch of values then adds as
// the sum of its integers, in any order and in parallel, plus its round-up
// bits, as long as this cannot carry the sum out of the binade; the integers
// stay below 2^53, where FP64 adds them exactly.  A batch that may leave the binade
// is cut into smaller ones, down to single additions.  (Halfway cases are common:
// a grid step with few significant bits gives coordinates on a lattice, and the
// unit of a long sum is a few lattice steps.)
#pragma once

#include <hip/hip_runtime.h>

namespace pp2p {

// 1 / u of the binade of s: 2^(52 - e) for |s| in [2^e, 2^(e+1)); 0 where the
// rule does not apply (zero, subnormal, infinite, NaN, or 1 / u out of range).
__host__ __device__ inline double seq_scale(double s)
{
    unsigned long long b;
    __builtin_memcpy(&b, &s, 8);
    const int be = (int)(b >> 52) & 0x7ff;              // biased exponent: e + 1023
    if (be < 60 || be > 1900)
        return 0.0;
    b = (unsigned long long)(1023 + 52 - (be - 1023)) << 52;
    double r;
    __builtin_memcpy(&r, &b, 8);
    return r;
}

// u itself from 1 / u: powers of two, whose exponents mirror each other
__host__ __device__ inline double seq_unit(double scale)
{
    unsigned long long b;
    __builtin_memcpy(&b, &scale, 8);
    b = (2046ull << 52) - b;
    double r;
    __builtin_memcpy(&r, &b, 8);
    return r;
}

// v in units of u: the nearest integer, or the lower one of a halfway case
// (half = true).  The product with a power of two is exact (or infinite, which
// fails the binade test below).
__host__ __device__ inline double seq_units(double v, double scale, bool &half)
{
    // q - r is exact (q - floor(q) is not: it rounds to 0.5 for q just above -0.5)
    const double q = v * scale, r = __builtin_rint(q);
    half = __builtin_fabs(q - r) == 0.5;
    return half ? __builtin_floor(q) : r;
}

__host__ __device__ inline bool seq_odd(double r)
{
    const double h = 0.5 * r;
    return h != __builtin_rint(h);
}

// parity of S, s in units of its binade: the last bit of its fraction
__host__ __device__ inline int seq_parity(double s)
{
    unsigned long long b;
    __builtin_memcpy(&b, &s, 8);
    return (int)(b & 1);
}

// The round-ups of a run of values as a function of the parity before it.
struct SeqTies {
    int any = 0;        // the run holds a halfway case
    int first = 0;      // round-up bit of the first one after an even S
    int rest = 0;       // round-ups of the later ones
    int out = 0;        // parity of S after the run: out, or parity before ^ out when !any
};

// round-ups of run t after parity p; p becomes the parity after it
__host__ __device__ inline int seq_roundups(const SeqTies &t, int &p)
{
    const int up = t.any ? (t.first ^ p) + t.rest : 0;
    p = t.any ? t.out : p ^ t.out;
    return up;
}

// Whether adding values whose units sum to up (those > 0) and down (the
// magnitudes of those < 0), in any order, keeps the sum S units strictly inside
// its binade; S > 0 (a negative sum is handled with every sign turned).  False
// for infinite or NaN sums.
__host__ __device__ inline bool seq_inside(double S, double up, double down)
{
    return S + up < 9007199254740992.0 && S - down > 4503599627370496.0;
}

}  // namespace pp2p
