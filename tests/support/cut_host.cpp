// Host build of the work-item cut search (photons-on-mt3000_amd/csrc/
// p2p_cut.h) for tests/test_cut_search.py and tests/test_cut_lanes.py: the
// search by one thread, and the device's by groups of 16 lanes of a wave, run on
// synthetic source-size prefixes at task indices up to 2^31 - 1, beside a
// sequential scan on exact 64-bit sums.  No device is used.
#include "../../photons-on-mt3000_amd/csrc/p2p_cut.h"

namespace {

// every source holds `size` particles: P(k) = k * size, modulo 2^32 as stored
struct ConstPrefix {
    unsigned size;
    unsigned operator()(int k) const { return (unsigned)((unsigned long long)k * size); }
};

// source j holds 1 + (7919 j mod 64) particles (1..64; a permutation of 1..64
// over each block of 64 consecutive j, so a block sums to 2080)
unsigned long long var_prefix_exact(long long k)
{
    unsigned long long s = (unsigned long long)(k / 64) * 2080ull;
    for (long long j = k - k % 64; j < k; ++j)
        s += 1ull + (unsigned long long)((7919ll * j) % 64);
    return s;
}

struct VarPrefix {
    unsigned operator()(int k) const { return (unsigned)var_prefix_exact(k); }
};

// A wave's groups of lanes search one row each, as the kernel does: every step
// all lanes of the groups that still search vote, and each group reads its own
// bits (the votes of a group that has ended are as its lanes' last).
template <class Prefix>
void wave_cuts(const Prefix &P, const int *beg, const int *end, long long wi, long long split, int *cut)
{
    constexpr int kGroups = 64 / pp2p::kCutLanes;
    for (int g = 0; g < kGroups; ++g) {
        const unsigned pb = P(beg[g]);
        cut[g] = pp2p::cut_search(beg[g], end[g], [&](long long lo, long long step, int n) {
            unsigned long long votes = 0;
            for (int lane = 0; lane < 64; ++lane) {
                const int j = lane % pp2p::kCutLanes, mine = lane / pp2p::kCutLanes;
                // the other groups' bits must not matter: all ones
                const bool over = mine == g ? pp2p::lane_over(P, pb, lo, step, n, j, wi, split) : true;
                votes |= (unsigned long long)over << lane;
            }
            return pp2p::first_over(votes, g * pp2p::kCutLanes, n);
        });
    }
}

}  // namespace

extern "C" {

// the cuts of the four rows [beg[g], end[g]) of a wave
void lanes_const(const int *beg, const int *end, long long wi, long long split, unsigned size, int *cut)
{
    wave_cuts(ConstPrefix{size}, beg, end, wi, split, cut);
}

void lanes_var(const int *beg, const int *end, long long wi, long long split, int *cut)
{
    wave_cuts(VarPrefix{}, beg, end, wi, split, cut);
}

int cut_const(int beg, int end, long long wi, long long split, unsigned size)
{
    return pp2p::range_cut(ConstPrefix{size}, beg, end, wi, split);
}

int cut_var(int beg, int end, long long wi, long long split)
{
    return pp2p::range_cut(VarPrefix{}, beg, end, wi, split);
}

// the first k in (beg, end] whose pairs of [beg, k] times wi exceed split, by
// a sequential scan on exact sums; end when none does
int cut_var_scan(int beg, int end, long long wi, long long split)
{
    const unsigned long long pb = var_prefix_exact(beg);
    for (long long k = beg + 1; k < end; ++k)
        if ((long long)(var_prefix_exact(k + 1) - pb) * wi > split)
            return (int)k;
    return end;
}

}  // extern "C"
