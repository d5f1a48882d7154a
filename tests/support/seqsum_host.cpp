// Host build of the parallel sequential sum (photons-on-mt3000_amd/csrc/
// p2p_seqsum.h) for tests/test_seqsum.py: batches accepted by the rule the tree
// kernels use, the others cut down to single additions, beside the plain
// loop.  No device is used.
#include "../../photons-on-mt3000_amd/csrc/p2p_seqsum.h"

#include <cmath>

namespace {

long long g_accepted;

double add_batch(double s, const double *v, long long n)
{
    const double scale = pp2p::seq_scale(s);
    if (scale != 0.0) {
        // the integers from the last value to the first: their order must not
        // matter; the round-ups in two runs, the first one's computed without the
        // parity before it
        double up = 0.0, down = 0.0;
        pp2p::SeqTies run[2];
        for (long long k = n - 1; k >= 0; --k) {
            bool half;
            const double r = pp2p::seq_units(v[k], s < 0.0 ? -scale : scale, half);
            (r > 0.0 ? up : down) += std::fabs(r);
        }
        for (long long k = 0; k < n; ++k) {
            bool half;
            const double r = pp2p::seq_units(v[k], s < 0.0 ? -scale : scale, half);
            pp2p::SeqTies &t = run[k >= n / 3];
            t.out ^= pp2p::seq_odd(r);
            if (half) {
                (t.any ? t.rest : t.first) += t.out;
                t.any = 1;
                t.out = 0;
            }
        }
        int p = pp2p::seq_parity(s), ups = 0;
        for (const pp2p::SeqTies &t : run)
            ups += pp2p::seq_roundups(t, p);
        up += ups;
        const double S = std::fabs(s) * scale;
        if (pp2p::seq_inside(S, up, down)) {
            g_accepted += n;
            const double m = (S + up - down) * pp2p::seq_unit(scale);
            return s < 0.0 ? -m : m;
        }
    }
    if (n == 1)
        return s + v[0];
    return add_batch(add_batch(s, v, n / 2), v + n / 2, n - n / 2);
}

}  // namespace

extern "C" {

double seqsum_batches(const double *v, long long n, long long batch, long long *accepted)
{
    double s = 0.0;
    g_accepted = 0;
    for (long long b = 0; b < n; b += batch)
        s = add_batch(s, v + b, n - b < batch ? n - b : batch);
    *accepted = g_accepted;
    return s;
}

double seqsum_loop(const double *v, long long n)
{
    volatile double s = 0.0;
    for (long long k = 0; k < n; ++k)
        s = s + v[k];
    return s;
}

}  // extern "C"
