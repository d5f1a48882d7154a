// Source-range cut of a CSR row, shared by the item-build kernels and the
// host (where it is tested at task indices beyond 2^30 and 2^31 - 1 without a
// device or a list of that size).
#pragma once

#include <hip/hip_runtime.h>

namespace pp2p {

// The cut after `beg` in a row whose tasks are [beg, end): the first k in
// (beg, end] with (pairs of tasks [beg, k]) * wi > split, or end when there
// is none.  P(k) is the exclusive prefix of the source sizes over the CSR
// modulo 2^32 (k = 0 .. ntask); differences within a row are exact.  The
// predicate grows with k, so probing kCutLanes even points at a time finds what
// a sequential scan would: two trips to memory for the usual row of a few
// hundred sources where halving takes eight.  Every P index lies in [beg, end];
// probes are formed in 64 bits (task indices pass 2^30).
constexpr int kCutLanes = 16;

// first(lo, step, n): the first of the n <= kCutLanes probes lo + (j + 1) step - 1
// that is over the limit, or n when none is.
template <class First>
__host__ __device__ inline int cut_search(int beg, int end, const First &first)
{
    long long lo = beg + 1ll, hi = end;
    while (lo < hi) {
        const long long step = (hi - lo + kCutLanes - 1) / kCutLanes;
        const int n = (int)((hi - lo) / step);          // probes below hi
        const int c = first(lo, step, n);
        if (c < n)
            hi = lo + (c + 1) * step - 1;
        lo += c * step;
    }
    return (int)lo;
}

template <class Prefix>
__host__ __device__ inline bool cut_over(const Prefix &P, unsigned pb, long long k, long long wi, long long split)
{
    return (long long)(P((int)(k + 1)) - pb) * wi > split;
}

// The form of kCutLanes lanes that search together: probe j, taken by lane j ...
template <class Prefix>
__host__ __device__ inline bool lane_over(const Prefix &P, unsigned pb, long long lo, long long step, int n, int j,
                                         long long wi, long long split)
{
    return j < n && cut_over(P, pb, lo + (j + 1) * step - 1, wi, split);
}

// ... and the first lane over the limit of the group that starts at lane `group`
// of the wave, n when none is (votes: one bit per lane of the wave).
__host__ __device__ inline int first_over(unsigned long long votes, int group, int n)
{
    const unsigned m = (unsigned)(votes >> group) & ((1u << kCutLanes) - 1u);
    return m ? __builtin_ctz(m) : n;
}

// one thread's form
template <class Prefix>
__host__ __device__ inline int range_cut(const Prefix &P, int beg, int end, long long wi, long long split)
{
    const unsigned pb = P(beg);
    return cut_search(beg, end, [&](long long lo, long long step, int n) {
        int j = 0;
        while (j < n && !cut_over(P, pb, lo + (j + 1) * step - 1, wi, split))
            ++j;
        return j;
    });
}

// The prefix as the device stores it: nsx[k].
struct PrefixArray {
    const unsigned *p;
    __host__ __device__ unsigned operator()(int k) const { return p[k]; }
};

}  // namespace pp2p
