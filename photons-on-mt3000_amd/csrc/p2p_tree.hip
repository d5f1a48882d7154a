// The kd-tree on the device: build_localtree's mean-split tree
// (src/fmm.c:168-270), its boxes (center_kdtree, src/fmm.c:273-327) and the
// target marking (src/fmm.c:1226-1236), with the reference's numbering and
// particle order.
//
// Segments (particle ranges) of more than kSubMax particles are split level by
// level over the whole device, the smaller ones each by one workgroup that
// keeps its particles in LDS and builds the whole subtree below them.  All
// segments at depth l split along coordinate l % 3.  A split:
//   mean    the sampled coordinates summed in FP64 in the reference's order
//           (stride len / 100000 above 10^5 particles), so the split is the
//           reference's to the bit; the additions run in parallel where their
//           rounding allows it (p2p_seqsum.h)
//   small   coordinate <= mean, as bit masks with their counts
//   swaps   the reference's in-place partition (src/fmm.c:199-219) scans
//           from the left for particles above the mean and swaps each with
//           the next particle at or below it from the right.  Its outcome
//           in closed form: with k particles at or below the mean, the i-th
//           particle above it in [0, k) is swapped with the i-th particle at
//           or below it counted from the end of [k, len); the left child
//           gets k particles, or len - 1 when every particle is at or below
//           the mean (the scan then stops one short).  Two particles are
//           ordered by a plain compare (src/fmm.c:180-187).
//   sons    more than maxleaf particles: a segment or subtree; else a leaf
// Afterwards the subtree sizes are summed bottom-up and the depth-first ids
// (nodes in creation order, leaves in creation order) and boxes handed
// top-down.  FP64 sums and FP32 boxes are rounded per operation (no
// contraction), as the host code computes them.
#include "p2p_seqsum.h"
#include "p2p_tree.h"

#pragma clang fp contract(off)

namespace pp2p {
namespace {

constexpr int kTreeBlock = 256;

inline unsigned grid_of(long long n) { return (unsigned)((n + kTreeBlock - 1) / kTreeBlock); }

// One workgroup per tile, segment or subtree: a grid holds fewer than 2^32 work
// items in x, 2^22 workgroups of 1024, and a tree with leaves of one particle has that
// many segments from 2^23 particles on.
inline dim3 wide_grid(long long blocks)
{
    constexpr long long kWide = 1 << 20;
    return blocks <= kWide ? dim3((unsigned)blocks) : dim3((unsigned)kWide, (unsigned)((blocks + kWide - 1) / kWide));
}

__device__ __forceinline__ int block_id() { return (int)(blockIdx.y * gridDim.x + blockIdx.x); }

__device__ __forceinline__ long long gid() { return (long long)blockIdx.x * kTreeBlock + threadIdx.x; }

__global__ __launch_bounds__(kTreeBlock) void k_tree_init(const int *__restrict__ posi, long long n,
                                                        TreeScratch w, TreeCounts *counts, TreeLevelView root,
                                                        TreeSub *sub)
{
    const long long i = gid();
    if (i == 0) {
        counts->nsub = sub ? 1 : 0;
        counts->misfit = 0;
        counts->nseg[0] = sub ? 0 : 1;
        if (sub) {
            sub[0].start = 0;
            sub[0].len = (int)n;
            sub[0].depth = 0;
        } else {
            root.seg[0] = make_int2(0, (int)n);
            root.toff[0] = 0;
            root.toff[1] = (int)((n + kTreeTile - 1) / kTreeTile);
        }
    }
    if (i >= n)
        return;
    w.x[0][i] = posi[3 * i];
    w.x[1][i] = posi[3 * i + 1];
    w.x[2][i] = posi[3 * i + 2];
    w.idx[i] = (int)i;
}

// ------------------------------------------------------------- exact sums

__device__ __forceinline__ double lane_value(double v, int k)
{
    const unsigned long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, k);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), k);
    return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

// Inclusive prefix sum over the wave by DPP (rows of 16, then the rows' totals
// handed on): six steps of two moves and an addition.  With __shfl_up (two LDS
// permutes per step) the subtrees of the 256^3 clustered tree took 3.9 ms
// instead of 3.3.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double v)
{
    const unsigned long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xf, true);
    return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

__device__ __forceinline__ double wave_prefix(double v)
{
    v += dpp_or_zero<0x111, 0xf>(v);                 // row_shr 1, 2, 4, 8
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    v += dpp_or_zero<0x142, 0xa>(v);                 // row_bcast 15 into rows 1 and 3
    v += dpp_or_zero<0x143, 0xc>(v);                 // row_bcast 31 into rows 2 and 3
    return v;
}

__device__ __forceinline__ double wave_sum(double v) { return lane_value(wave_prefix(v), 63); }

// A lane's kV consecutive values as units of s's binade: their sums by sign,
// and their round-ups, which are zero without a halfway case.
template <int kV>
__device__ __forceinline__ SeqTies lane_units(const double (&v)[kV], double scale, double &up, double &down)
{
    SeqTies run;
    up = down = 0.0;
#pragma unroll
    for (int u = 0; u < kV; ++u) {
        bool half;
        const double r = seq_units(v[u], scale, half);
        up += r > 0.0 ? r : 0.0;
        down += r < 0.0 ? -r : 0.0;
        run.out ^= seq_odd(r);
        if (half) {
            (run.any ? run.rest : run.first) += run.out;
            run.any = 1;
            run.out = 0;
        }
    }
    return run;
}

// Parity before each lane's run when it is p before the first lane's; `all`
// (the same in every lane) becomes the runs of all lanes as one, but for its
// rest, which is each lane's share.
__device__ __forceinline__ int lanes_parity(const SeqTies &run, int p, int lane, SeqTies &all)
{
    const unsigned long long outs = __ballot(run.out), any = __ballot(run.any);
    const unsigned long long upto = ~0ull >> (63 - lane);
    const int c = __popcll(outs & upto) & 1;         // parity of the outs up to and with this lane's
    all.out = __popcll(outs) & 1;
    if (!any) {
        all.any = all.first = all.rest = 0;
        return p ^ c ^ run.out;
    }
    const unsigned long long cs = __ballot(c), prev = any & (upto >> 1);
    // outs of the lanes after the last halfway case's, and its own parity
    auto since = [&](int k) { return (int)(cs >> k) ^ (int)(outs >> k); };
    const int l = 63 - __clzll(any), f = __builtin_ctzll(any);
    const int before = prev ? (c ^ run.out ^ since(63 - __clzll(prev))) & 1 : p ^ c ^ run.out;
    const int first = __builtin_amdgcn_readlane(run.first, f) ^ ((int)((cs ^ outs) >> f) & 1);
    all.any = 1;
    all.first = first & 1;                           // with parity 0 before the first lane
    all.rest = run.any ? run.rest + (lane != f ? run.first ^ before : 0) : 0;
    all.out = (all.out ^ since(l)) & 1;
    return before;
}

// s + the first cnt of a wave's 64 values, one after the other, the same in every
// lane: 16 to 20 cycles a value, so 64 values cost less than the passes of add_run
// that a group which leaves its binade needs (about 2 us).
__device__ __forceinline__ double add_chain(double s, double v, int cnt)
{
    constexpr int kStep = 16;
    if (cnt >= 64) {
#pragma unroll
        for (int k = 0; k < 64; ++k)
            s += lane_value(v, k);
        return s;
    }
    for (int k = 0; k < cnt; k += kStep)             // (+0.0 past the end)
#pragma unroll
        for (int u = 0; u < kStep; ++u)
            s += lane_value(v, k + u);
    return s;
}

// s + a wave's 64 kV values, lane l's before lane l + 1's, the same in every
// lane.  A pass adds the lanes up to the first whose values may leave the sum's
// binade by one prefix sum, then that lane's one after the other.  A sum from zero
// starts with eight lanes' values one after the other, where the binades are
// short.
template <int kV>
__device__ double add_run(double s, const double (&v)[kV], int lane)
{
    auto serial = [&](int l) {
#pragma unroll
        for (int u = 0; u < kV; ++u)
            s += lane_value(v[u], l);
    };
    int next = 0;
    while (next < 64) {
        const double scale = seq_scale(s);
        if (scale == 0.0) {
            const int e = next == 0 ? 8 : next + 1;
            for (; next < e; ++next)
                serial(next);
            continue;
        }
        double up, down;
        SeqTies run = lane_units(v, s < 0.0 ? -scale : scale, up, down), all;
        if (lane < next) {
            up = down = 0.0;
            run = SeqTies();
        }
        if (__ballot(run.any)) {
            int p = lanes_parity(run, seq_parity(s), lane, all);
            up += (double)seq_roundups(run, p);
        }
        const double S = fabs(s) * scale, inc = up - down;
        const double t = wave_prefix(inc);
        const unsigned long long bad = __ballot(!seq_inside(S + (t - inc), up, down)) & (~0ull << next);
        const int first = bad ? __builtin_ctzll(bad) : 64;
        if (first > next) {
            const double m = (S + lane_value(t, first - 1)) * seq_unit(scale);
            s = s < 0.0 ? -m : m;
        }
        if (first < 64)
            serial(first);
        next = first + 1;
    }
    return s;
}

// Sums of long segments take three steps, so that all but the last run in
// parallel: plain sums of groups of 64 values say in which binade each group
// starts (nearly always; a wrong guess only costs time), every group is turned
// into units of that binade, and one wave composes the groups in order, 64 at a
// time by a prefix sum.  A group that leaves its binade or was guessed wrong is
// added by itself from its values.
constexpr int kGroup = 64;

// info: 0 where the rule does not apply, else the start's sign and exponent
// (bits 11 to 22) and the SeqTies of the group (any, first, out, rest)
struct GroupUnits {
    double up, down;
    int info;
};

__device__ __forceinline__ int binade_of(double s)
{
    return seq_scale(s) == 0.0 ? 0 : (int)((unsigned long long)__double_as_longlong(s) >> 52) << 11;
}

// The wave's 64 values (+0.0 past the end) as units of the binade of `start`.
__device__ __forceinline__ GroupUnits group_units(double v, double start, int lane)
{
    GroupUnits g{0.0, 0.0, binade_of(start)};
    if (!g.info)
        return g;
    const double scale = seq_scale(start), one[1] = {v};
    const SeqTies run = lane_units(one, start < 0.0 ? -scale : scale, g.up, g.down);
    SeqTies all;
    if (__ballot(run.any)) {
        lanes_parity(run, 0, lane, all);
        all.rest = __popcll(__ballot(all.rest));
    } else {
        all.out = __popcll(__ballot(run.out)) & 1;
    }
    g.up = __ballot(g.up != 0.0) ? wave_sum(g.up) : 0.0;
    g.down = __ballot(g.down != 0.0) ? wave_sum(g.down) : 0.0;
    g.info |= all.any | all.first << 1 | all.out << 2 | all.rest << 3;
    return g;
}

// s + the cnt <= 64 groups from `base` on, the same in every lane: u is the
// lane's group, value(g) the lane's value of group g.
template <class Value>
__device__ __forceinline__ double add_groups(double s, const GroupUnits &u, int base, int cnt, int lane, Value value)
{
    int next = 0;
    while (next < cnt) {
        const double scale = seq_scale(s), S = fabs(s) * scale;
        const int at = binade_of(s);
        const bool mine = lane >= next && lane < cnt && at && (u.info >> 11) == (at >> 11);
        SeqTies run, all;
        double up = 0.0, down = 0.0;
        if (mine) {
            run.any = u.info & 1;
            run.first = u.info >> 1 & 1;
            run.out = u.info >> 2 & 1;
            run.rest = u.info >> 3 & 0xff;
            up = u.up;
            down = u.down;
        }
        int p = lanes_parity(run, seq_parity(s), lane, all);
        up += (double)seq_roundups(run, p);
        const double inc = up - down, t = wave_prefix(inc);
        const unsigned long long bad =
            __ballot(!mine || !seq_inside(S + (t - inc), up, down)) & (~0ull << next) & (~0ull >> (64 - cnt));
        const int first = bad ? __builtin_ctzll(bad) : cnt;
        if (first > next) {
            const double m = (S + lane_value(t, first - 1)) * seq_unit(scale);
            s = s < 0.0 ? -m : m;
        }
        if (first < cnt)
            s = add_chain(s, value(base + first), 64);
        next = first + 1;
    }
    return s;
}

// Plain sums: they only say where a group is expected to start.
__device__ __forceinline__ float wave_sum_about(float v)
{
    auto step = [&](int moved) { v += __int_as_float(moved); };
    const auto bits = [&] { return __float_as_int(v); };
    step(__builtin_amdgcn_update_dpp(0, bits(), 0x111, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, bits(), 0x112, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, bits(), 0x114, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, bits(), 0x118, 0xf, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, bits(), 0x142, 0xa, 0xf, true));
    step(__builtin_amdgcn_update_dpp(0, bits(), 0x143, 0xc, 0xf, true));
    return __int_as_float(__builtin_amdgcn_readlane(bits(), 63));
}

// ------------------------------------------------------------- level passes

// the segment holding a tile: the last s with toff[s] <= tile
__device__ __forceinline__ int seg_of_tile(const int *__restrict__ toff, int nseg, int tile)
{
    int lo = 0, hi = nseg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (toff[mid] <= tile)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Split values (src/fmm.c:168-197): the sampled FP64 mean for more than two
// particles, the midpoint of two, 0 for fewer.  A segment's samples (all
// particles, or every (len / 10^5)-th) in chunks of 4096: sums of the chunks, the
// groups of each chunk in units, and one wave per segment that composes them.
// The first two are bound by HBM, the last by the chain of about ten groups that
// change the binade, 1 us each with the load of their samples (2 with add_run in
// place of a plain chain: 9 levels of 64^3 280 -> 199 us, 18 of 256^3 890 -> 720).  One workgroup
// per segment doing all of it, one 4096 values after the other, was bound by
// the loads and the rounding of a single CU where the segments are few: 9 levels of
// 64^3 took 625 us and take 315, 18 of 256^3 (clustered) 2500 and take 1700.
struct Samples {
    const int *x;                                    // the segment's coordinates
    long long mul;
    int ns, chunks;
    double int2pos;
    __device__ Samples(const int *coord, int2 seg, double step) : x(coord + seg.x), mul(1), int2pos(step)
    {
        if (seg.y > 100000)
            mul = seg.y / 100000;
        ns = seg.y > 2 ? (int)((seg.y + mul - 1) / mul) : 0;
        chunks = (ns + kTreeTile - 1) / kTreeTile;   // at most 49, and at most the segment's tiles
    }
    // sample k, +0.0 past the end
    __device__ double operator()(int k) const
    {
        const int r = x[(k < ns ? k : ns - 1) * mul];
        return k < ns ? int2pos * (double)r : 0.0;
    }
};

// plain sums of the chunks; tmap[tile] = the tile's segment
__global__ __launch_bounds__(kTreeBlock) void k_tree_sums(TreeLevelView lv, const int *__restrict__ nseg,
                                                        const int *__restrict__ x, double int2pos,
                                                        double *__restrict__ csum, int *__restrict__ tmap)
{
    __shared__ double part[kTreeBlock / 64];
    const int n = *nseg, tile = block_id();
    if (n == 0 || tile >= lv.toff[n])
        return;
    const int s = seg_of_tile(lv.toff, n, tile);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0)
        tmap[tile] = s;
    const Samples v(x, lv.seg[s], int2pos);
    const int c = tile - lv.toff[s];
    if (c >= v.chunks)
        return;
    double sum = 0.0;
#pragma unroll
    for (int u = 0; u < kTreeTile / kTreeBlock; ++u)
        sum += v(c * kTreeTile + u * kTreeBlock + (int)threadIdx.x);
    sum = wave_sum(sum);
    if (lane == 0)
        part[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < kTreeBlock / 64; ++q)
            sum += part[q];
        csum[tile] = sum;
    }
}

// the groups of each chunk in units
constexpr int kUnitBlock = 1024;

__global__ __launch_bounds__(kUnitBlock) void k_tree_units(TreeLevelView lv, const int *__restrict__ nseg,
                                                         const int *__restrict__ x, double int2pos,
                                                         const double *__restrict__ csum,
                                                         const int *__restrict__ tmap,
                                                         GroupUnits *__restrict__ units)
{
    constexpr int kGroups = kTreeTile / kGroup, kPerWave = kGroups / (kUnitBlock / 64);
    __shared__ double start[kGroups];
    const int n = *nseg, tile = block_id();
    if (n == 0 || tile >= lv.toff[n])
        return;
    const int s = tmap[tile];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const Samples v(x, lv.seg[s], int2pos);
    const int t0 = lv.toff[s], c = tile - t0;
    if (c >= v.chunks)
        return;
    double mine[kPerWave];
#pragma unroll
    for (int u = 0; u < kPerWave; ++u)
        mine[u] = v(c * kTreeTile + (wave * kPerWave + u) * kGroup + lane);
#pragma unroll
    for (int u = 0; u < kPerWave; ++u) {
        const float g = wave_sum_about((float)mine[u]);
        if (lane == 0)
            start[wave * kPerWave + u] = (double)g;
    }
    __syncthreads();
    if (wave == 0) {
        const double before = wave_sum(lane < c ? csum[t0 + lane] : 0.0);
        const double g = start[lane];
        start[lane] = before + (wave_prefix(g) - g);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPerWave; ++u) {
        const int g = wave * kPerWave + u;
        const GroupUnits r = group_units(mine[u], start[g], lane);
        if (lane == 0)
            units[(long long)tile * kGroups + g] = r;
    }
}

constexpr int kAhead = 4;                            // batches of groups loaded together

__global__ __launch_bounds__(64) void k_tree_mean(TreeLevelView lv, const int *__restrict__ nseg,
                                                const int *__restrict__ x, double int2pos,
                                                const GroupUnits *__restrict__ units)
{
    const int s = block_id(), lane = threadIdx.x;
    if (s >= *nseg)
        return;
    const int2 sg = lv.seg[s];
    const Samples v(x, sg, int2pos);
    double m = 0.0;
    float sp = 0.0f;
    if (sg.y > 2) {
        const GroupUnits *u = units + (long long)lv.toff[s] * (kTreeTile / kGroup);
        const int ng = (v.ns + kGroup - 1) / kGroup;
        for (int base = 0; base < ng; base += kAhead * 64) {
            GroupUnits r[kAhead];                    // loads in flight together
#pragma unroll
            for (int q = 0; q < kAhead; ++q)
                r[q] = u[min(base + q * 64 + lane, ng - 1)];
#pragma unroll
            for (int q = 0; q < kAhead; ++q)
                m = add_groups(m, r[q], base + q * 64, min(64, ng - base - q * 64), lane,
                               [&](int g) { return v(g * kGroup + lane); });
        }
        m /= (double)sg.y;
        m *= (double)v.mul;
        sp = (float)m;
    } else if (sg.y == 2) {
        sp = (float)(0.5 * (int2pos * (double)(x[sg.x] + x[sg.x + 1])));
    }
    if (lane == 0) {
        lv.mean[s] = m;
        lv.split[s] = sp;
    }
}

// Masks of the particles at or below the mean, 64 words and their total per
// tile of kTreeTile positions of one segment.
__global__ __launch_bounds__(kTreeBlock) void k_tree_flags(TreeLevelView lv, const int *__restrict__ nseg,
                                                         const int *__restrict__ x, double int2pos,
                                                         unsigned long long *__restrict__ mask,
                                                         int *__restrict__ tcnt, const int *__restrict__ tmap)
{
    __shared__ int part[kTreeBlock / 64];
    const int ns = *nseg, tile = block_id();
    if (ns == 0 || tile >= lv.toff[ns])
        return;
    const int s = tmap[tile];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int2 sg = lv.seg[s];
    const double mean = lv.mean[s];
    const int base = (tile - lv.toff[s]) * kTreeTile;     // offset of the tile in its segment
    constexpr int kWords = kTreeTile / kTreeBlock;        // words per wave
    int r[kWords];
#pragma unroll
    for (int u = 0; u < kWords; ++u) {
        const int p = base + (wave * kWords + u) * 64 + lane;
        r[u] = p < sg.y ? x[sg.x + p] : 0;
    }
    int cnt = 0;
    unsigned long long keep = 0;
#pragma unroll
    for (int u = 0; u < kWords; ++u) {
        const int p = base + (wave * kWords + u) * 64 + lane;
        const unsigned long long m = __ballot(p < sg.y && sg.y > 2 && !(int2pos * (double)r[u] > mean));
        if (lane == u)
            keep = m;
        cnt += __popcll(m);
    }
    if (lane < kWords)
        mask[(long long)tile * (kTreeTile / 64) + wave * kWords + lane] = keep;
    if (lane == 0)
        part[wave] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int q = 0; q < kTreeBlock / 64; ++q)
            t += part[q];
        tcnt[tile] = t;
    }
}

// The misplaced particles of each segment by rank: la[a + r] = the r-th
// particle above the mean in the left part, lb[a + r] = the r-th at or below it
// counted from the end of the right part; the left son's size and the
// number of swaps.  A tile finds the counts before it by summing the tile
// counts of its segment (at most n / 4096 integers from L2).
__global__ __launch_bounds__(kTreeBlock) void k_tree_lists(TreeLevelView lv, const int *__restrict__ nseg,
                                                         const int *__restrict__ x,
                                                         const unsigned long long *__restrict__ mask,
                                                         const int *__restrict__ tcnt,
                                                         const int *__restrict__ tmap, int *__restrict__ la,
                                                         int *__restrict__ lb)
{
    constexpr int kWords = kTreeTile / 64;
    __shared__ int before_s[kTreeBlock / 64], total_s[kTreeBlock / 64];
    __shared__ unsigned long long word[kWords];
    __shared__ int wpre[kWords];
    const int ns = *nseg, tile = block_id();
    if (ns == 0 || tile >= lv.toff[ns])
        return;
    const int s = tmap[tile];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int a = lv.seg[s].x, len = lv.seg[s].y;
    const int t0 = lv.toff[s], t1 = lv.toff[s + 1];
    if (len <= 2) {                                  // one tile
        if (threadIdx.x == 0) {
            const bool sw = len == 2 && x[a] > x[a + 1];
            lv.left[s] = len == 2 ? 1 : 0;
            lv.swaps[s] = sw;
            if (sw) {
                la[a] = a;
                lb[a] = a + 1;
            }
        }
        return;
    }
    int before = 0, total = 0;
    for (int t = t0 + (int)threadIdx.x; t < t1; t += kTreeBlock) {
        const int c = tcnt[t];
        total += c;
        before += t < tile ? c : 0;
    }
    for (int o = 32; o > 0; o >>= 1) {
        before += __shfl_xor(before, o, 64);
        total += __shfl_xor(total, o, 64);
    }
    if (lane == 0) {
        before_s[wave] = before;
        total_s[wave] = total;
    }
    if (wave == 0) {
        const unsigned long long m = mask[(long long)tile * kWords + lane];
        const int c = __popcll(m);
        int inc = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc, o, 64);
            if (lane >= o)
                inc += u;
        }
        word[lane] = m;
        wpre[lane] = inc - c;
    }
    __syncthreads();
    before = total = 0;
    for (int q = 0; q < kTreeBlock / 64; ++q) {
        before += before_s[q];
        total += total_s[q];
    }
    if (total == len) {
        if (tile == t0 && threadIdx.x == 0) {
            lv.left[s] = len - 1;
            lv.swaps[s] = 0;
        }
        return;
    }
    const int k = total;
    if (tile == t0 && threadIdx.x == 0)
        lv.left[s] = k;
    const int base = (tile - t0) * kTreeTile;
    for (int o = threadIdx.x; o < kTreeTile; o += kTreeBlock) {
        const int p = base + o;
        if (p >= len)
            break;
        const unsigned long long m = word[o >> 6];
        const int sb = before + wpre[o >> 6] + __popcll(m & ((1ull << (o & 63)) - 1ull));   // small ones before p
        const bool small = (m >> (o & 63)) & 1ull;
        if (p == k)
            lv.swaps[s] = k - sb;                    // k < len here: exactly one thread of the segment
        if (p < k && !small)
            la[a + (p - sb)] = a + p;
        else if (p >= k && small)
            lb[a + (k - sb - 1)] = a + p;
    }
}

__device__ __forceinline__ void swap_part(int *x0, int *x1, int *x2, int *idx, int i, int j)
{
    const int a0 = x0[i], a1 = x1[i], a2 = x2[i], a3 = idx[i];
    const int b0 = x0[j], b1 = x1[j], b2 = x2[j], b3 = idx[j];
    x0[i] = b0; x1[i] = b1; x2[i] = b2; idx[i] = b3;
    x0[j] = a0; x1[j] = a1; x2[j] = a2; idx[j] = a3;
}

// The partition's swaps, in place: each swapped pair belongs to one thread.
// Bound by HBM: 32 B read and written per pair and 8 B of lists; the level passes
// together took 363 us per level on the 256^3 clustered tree when each ran
// over every particle with its segment looked up per particle.
__global__ __launch_bounds__(kTreeBlock) void k_tree_swap(TreeLevelView lv, const int *__restrict__ nseg,
                                                        const int *__restrict__ tmap, TreeScratch w)
{
    const int ns = *nseg, tile = block_id();
    if (ns == 0 || tile >= lv.toff[ns])
        return;
    const int s = tmap[tile];
    const int a = lv.seg[s].x, r0 = (tile - lv.toff[s]) * kTreeTile;
    const int r1 = min(r0 + kTreeTile, lv.swaps[s]);
    for (int r = r0 + (int)threadIdx.x; r < r1; r += kTreeBlock)
        swap_part(w.x[0], w.x[1], w.x[2], w.idx, w.la[a + r], w.lb[a + r]);
}

// The sons of a level, in order: the next level's segments with their tile
// offsets, the new subtrees, this level's leaves.  One block: a level holds at
// most n / kSubMax segments.
constexpr int kNextBlock = 1024;

__global__ __launch_bounds__(kNextBlock) void k_tree_next(TreeLevelView lv, TreeLevelView nx, int level, int maxleaf,
                                                        int gmax, TreeCounts *counts, TreeSub *sub, int subcap)
{
    __shared__ int4 wtot[kNextBlock / 64];
    const int ns = counts->nseg[level];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int4 base = make_int4(0, counts->nsub, 0, 0);    // next segments, subtrees, leaves, tiles
    __syncthreads();                                 // every thread has read nsub before it changes
    for (int b = 0; b < ns; b += kNextBlock) {
        const int s = b + (int)threadIdx.x;
        int rs[2] = {0, 0}, rn[2] = {0, 0}, kind[2] = {-1, -1};
        int4 c = make_int4(0, 0, 0, 0);
        if (s < ns) {
            const int2 sg = lv.seg[s];
            const int l = lv.left[s];
            rs[0] = sg.x; rn[0] = l;
            rs[1] = sg.x + l; rn[1] = sg.y - l;
            for (int h = 0; h < 2; ++h) {
                kind[h] = rn[h] > gmax ? 0 : rn[h] > maxleaf ? 1 : 2;
                c.x += kind[h] == 0;
                c.y += kind[h] == 1;
                c.z += kind[h] == 2;
                c.w += kind[h] == 0 ? (rn[h] + kTreeTile - 1) / kTreeTile : 0;
            }
        }
        int4 inc = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int4 u = make_int4(__shfl_up(inc.x, o, 64), __shfl_up(inc.y, o, 64), __shfl_up(inc.z, o, 64),
                                     __shfl_up(inc.w, o, 64));
            if (lane >= o) {
                inc.x += u.x; inc.y += u.y; inc.z += u.z; inc.w += u.w;
            }
        }
        if (lane == 63)
            wtot[wave] = inc;
        __syncthreads();
        int4 at = make_int4(base.x + inc.x - c.x, base.y + inc.y - c.y, base.z + inc.z - c.z, base.w + inc.w - c.w);
        for (int q = 0; q < kNextBlock / 64; ++q) {
            const int4 t = wtot[q];
            if (q < wave) {
                at.x += t.x; at.y += t.y; at.z += t.z; at.w += t.w;
            }
            base.x += t.x; base.y += t.y; base.z += t.z; base.w += t.w;
        }
        __syncthreads();                             // wtot is rewritten by the next chunk
        if (s < ns) {
            int code[2];
            for (int h = 0; h < 2; ++h) {
                const int2 rg = make_int2(rs[h], rn[h]);
                if (kind[h] == 0) {
                    nx.seg[at.x] = rg;
                    nx.toff[at.x] = at.w;
                    at.w += (rn[h] + kTreeTile - 1) / kTreeTile;
                    code[h] = at.x++;
                } else if (kind[h] == 1) {
                    if (at.y < subcap) {
                        sub[at.y].start = rg.x;
                        sub[at.y].len = rg.y;
                        sub[at.y].depth = level + 1;
                    } else {
                        counts->misfit = 1;
                    }
                    code[h] = kSubKid + at.y++;
                } else {
                    lv.leaf[at.z] = rg;
                    code[h] = -at.z++ - 1;
                }
            }
            lv.kid[s] = make_int2(code[0], code[1]);
        }
    }
    if (threadIdx.x == 0) {
        counts->nsub = base.y < subcap ? base.y : subcap;
        counts->nseg[level + 1] = base.x;
        nx.toff[base.x] = base.w;
    }
}

// ------------------------------------------------------------- subtrees

// A whole subtree of at most kSubMax particles by one workgroup, the particles
// in LDS from the first split to the last.  Per level: the means (one thread
// per segment from eight on, one wave per segment otherwise), the masks, the partners, the swaps, the sons.  The nodes are
// numbered breadth first while they are made and depth first at the end.
// Bound by the latencies of about eight levels (the means first, then seven
// barriers each); it takes the place of as many passes over all particles in
// HBM: 2.6 ms for 1.9 10^7 particles (256^3 clustered; 3.0 with add_run for all
// levels of fewer than 48 segments) where ten levels of device-wide passes took
// about 8.  4096 particles with the records fill one
// CU's LDS.  The whole build, uploads included, went from 28.2 to 15.7 ms
// there, from 4.6 to 1.5 ms at 64^3 and from 1.5 to 0.58 ms at 16^3.
constexpr int kSubBlock = 1024;
constexpr int kBatch = 8;            // values of a thread's chain loaded together
// How a level's segments are summed.  The parallel form (add_run) costs about
// 2 us for each change of the binade and, with several waves on a SIMD, the
// instructions of each; a plain chain costs its length.  Level by level of a subtree
// of 3200 particles (segments of 3200, 1600, ...): add_run 15 to 25, 10 to 20, 7 to
// 15, 13, 25 and 11 us; one wave's chain (segments of at most kSubChain) 9 us for
// 800 values, 7 for 400; one thread per segment, 14 ns a value, 11 for 800, then
// 6, 3.3 and 2.  With eight segments or more a level is as long as a thread's chain.
constexpr int kSubChain = 1024;
constexpr int kSubThreads = 8;

struct SubLds {
    int x[3][kSubMax], idx[kSubMax];
    unsigned short seg[kSubMax];                     // segment of the position (0xffff: in a leaf)
    unsigned short partner[kSubMax];
    unsigned long long mask[kSubMax / 64];
    int wpre[kSubMax / 64 + 1];
    unsigned short beg[2][kSubMax / 2], len[2][kSubMax / 2];
    double mean[kSubMax / 2];
    unsigned short left[kSubMax / 2], k[kSubMax / 2];    // k = 0xffff: no swaps
    short kid[2][kSubMax];                           // by node, breadth first: node >= 0, leaf -(q + 1)
    unsigned short lbeg[kSubMax], llen[kSubMax];     // leaves in creation order
    int nnext, nleaf, misfit;
};
static_assert(sizeof(SubLds) <= 160 * 1024, "one CU's LDS");
// the numbering reuses the particles' space
struct SubNumber {
    unsigned short nodes[kSubMax], leaves[kSubMax];  // below each node
    unsigned short id[kSubMax], leaf0[kSubMax];
    unsigned short up[kSubMax];                      // parent << 1 | side
};
static_assert(sizeof(GroupUnits) * (kTreeTile / kGroup) == kTreeUnitBytes, "tile record");
static_assert(sizeof(SubNumber) <= sizeof(SubLds::x), "numbering overlaps more than the coordinates");

__device__ __forceinline__ int sub_small_before(const SubLds &m, int p)
{
    const int w = p >> 6;
    return m.wpre[w] + ((p & 63) ? __popcll(m.mask[w] & ((1ull << (p & 63)) - 1ull)) : 0);
}

__global__ __launch_bounds__(kSubBlock) void k_tree_sub(TreeScratch w, TreeSub *__restrict__ sub, int nsub,
                                                      double int2pos, int maxleaf,
                                                      unsigned short *__restrict__ off_all, TreeCounts *counts)
{
    __shared__ SubLds m;
    if (block_id() >= nsub)
        return;
    TreeSub &me = sub[block_id()];
    unsigned short *off = off_all + (size_t)block_id() * kSubLevels;
    const int start = me.start, n = me.len, depth = me.depth;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < kSubMax; i += kSubBlock) {
        const bool in = i < n;
        m.x[0][i] = in ? w.x[0][start + i] : 0;
        m.x[1][i] = in ? w.x[1][start + i] : 0;
        m.x[2][i] = in ? w.x[2][start + i] : 0;
        m.idx[i] = in ? w.idx[start + i] : 0;
        m.seg[i] = in ? 0 : 0xffff;
    }
    if (tid == 0) {
        m.beg[0][0] = 0;
        m.len[0][0] = (unsigned short)n;
        m.nleaf = 0;
        m.misfit = 0;
        off[0] = 0;
    }
    __syncthreads();
    int nseg = 1, first = 0, lev = 0, cur = 0;       // first: breadth-first number of the level's first node
    // nodes and leaves have room for as many as the subtree has particles
    while (nseg > 0) {
        const int axis = (depth + lev) % 3;
        const int *x = m.x[axis];
        const unsigned short *beg = m.beg[cur], *slen = m.len[cur];
        // means and split values
        if (nseg >= kSubThreads) {
            for (int s = tid; s < nseg; s += kSubBlock) {
                const int b = beg[s], l = slen[s];
                double sum = 0.0;
                float sp = 0.0f;
                if (l > 2) {
                    int j = 0;
                    if (l >= kBatch) {               // the next batch is read ahead of this one's chain
                        int r[kBatch];
#pragma unroll
                        for (int q = 0; q < kBatch; ++q)
                            r[q] = x[b + q];
                        for (; j + 2 * kBatch <= l; j += kBatch) {
                            int ahead[kBatch];
#pragma unroll
                            for (int q = 0; q < kBatch; ++q)
                                ahead[q] = x[b + j + kBatch + q];
#pragma unroll
                            for (int q = 0; q < kBatch; ++q)
                                sum += int2pos * (double)r[q];
#pragma unroll
                            for (int q = 0; q < kBatch; ++q)
                                r[q] = ahead[q];
                        }
#pragma unroll
                        for (int q = 0; q < kBatch; ++q)
                            sum += int2pos * (double)r[q];
                        j += kBatch;
                    }
                    for (; j < l; ++j)
                        sum += int2pos * (double)x[b + j];
                    sum /= (double)l;
                    sp = (float)sum;
                } else if (l == 2) {
                    sp = (float)(0.5 * (int2pos * (double)(x[b] + x[b + 1])));
                }
                m.mean[s] = sum;
                w.lc[start + first + s] = __float_as_int(sp);
            }
        } else {
            for (int s = wave; s < nseg; s += kSubBlock / 64) {
                const int b = beg[s], l = slen[s];
                double sum = 0.0;
                float sp = 0.0f;
                if (l > 2 && l <= kSubChain) {
                    auto value = [&](int j) { return j < l ? int2pos * (double)x[b + j] : 0.0; };
                    double v = value(lane);
                    for (int c = 0; c < l; c += 64) {
                        const double ahead = value(c + 64 + lane);
                        sum = add_chain(sum, v, min(l - c, 64));
                        v = ahead;
                    }
                    sum /= (double)l;
                    sp = (float)sum;
                } else if (l > 2) {
                    for (int c = 0; c < l; c += 512) {
                        double v[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const int j = c + lane * 8 + u;
                            v[u] = j < l ? int2pos * (double)x[b + (j < l ? j : 0)] : 0.0;
                        }
                        sum = add_run(sum, v, lane);
                    }
                    sum /= (double)l;
                    sp = (float)sum;
                } else if (l == 2) {
                    sp = (float)(0.5 * (int2pos * (double)(x[b] + x[b + 1])));
                }
                if (lane == 0) {
                    m.mean[s] = sum;
                    w.lc[start + first + s] = __float_as_int(sp);
                }
            }
        }
        if (tid == 0)
            m.nnext = 0;
        __syncthreads();
        // masks of the particles at or below the mean
#pragma unroll
        for (int u = 0; u < kSubMax / kSubBlock; ++u) {
            const int wd = wave * (kSubMax / kSubBlock) + u, i = wd * 64 + lane;
            const int s = m.seg[i];
            const bool f = s != 0xffff && slen[s == 0xffff ? 0 : s] > 2 &&
                           !(int2pos * (double)x[i] > m.mean[s == 0xffff ? 0 : s]);
            const unsigned long long b = __ballot(f);
            if (lane == 0)
                m.mask[wd] = b;
        }
        __syncthreads();
        if (wave == 0) {
            const int c = __popcll(m.mask[lane]);
            int inc = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(inc, o, 64);
                if (lane >= o)
                    inc += u;
            }
            m.wpre[lane] = inc - c;
            if (lane == 63)
                m.wpre[64] = inc;
        }
        __syncthreads();
        auto before = [&](int p) { return p == kSubMax ? m.wpre[64] : sub_small_before(m, p); };
        for (int s = tid; s < nseg; s += kSubBlock) {
            const int b = beg[s], l = slen[s];
            int left = l == 2 ? 1 : 0, k = 0xffff;
            if (l > 2) {
                const int sm = before(b + l) - before(b);
                left = sm == l ? l - 1 : sm;
                k = sm == l ? 0xffff : sm;
            }
            m.left[s] = (unsigned short)left;
            m.k[s] = (unsigned short)k;
        }
        __syncthreads();
        // partners from the right part
        for (int i = tid; i < n; i += kSubBlock) {
            const int s = m.seg[i];
            if (s == 0xffff || m.k[s] == 0xffff || !((m.mask[i >> 6] >> (i & 63)) & 1ull))
                continue;
            const int b = beg[s];
            if (i >= b + m.k[s])
                m.partner[b + (m.k[s] - (before(i + 1) - before(b)))] = (unsigned short)i;
        }
        __syncthreads();
        for (int i = tid; i < n; i += kSubBlock) {
            const int s = m.seg[i];
            if (s == 0xffff)
                continue;
            const int b = beg[s];
            int j = -1;
            if (slen[s] == 2) {
                if (i == b && x[b] > x[b + 1])
                    j = b + 1;
            } else if (m.k[s] != 0xffff && i < b + m.k[s] && !((m.mask[i >> 6] >> (i & 63)) & 1ull)) {
                j = m.partner[b + (i - b) - (before(i) - before(b))];
            }
            if (j >= 0)
                swap_part(m.x[0], m.x[1], m.x[2], m.idx, i, j);
        }
        // sons: their breadth-first numbers in any order
        const int nfirst = first + nseg;
        for (int s = tid; s < nseg; s += kSubBlock) {
            const int b = beg[s], l = slen[s], left = m.left[s];
            for (int h = 0; h < 2; ++h) {
                const int cb = h ? b + left : b, cl = h ? l - left : left;
                int code = 0;
                if (cl > maxleaf) {
                    const int k = atomicAdd(&m.nnext, 1);
                    if (nfirst + k < n) {
                        m.beg[cur ^ 1][k] = (unsigned short)cb;
                        m.len[cur ^ 1][k] = (unsigned short)cl;
                        code = nfirst + k;
                    } else {
                        m.misfit = 1;
                    }
                } else {
                    const int q = atomicAdd(&m.nleaf, 1);
                    if (q < n) {
                        m.lbeg[q] = (unsigned short)cb;
                        m.llen[q] = (unsigned short)cl;
                        code = -q - 1;
                    } else {
                        m.misfit = 1;
                    }
                }
                m.kid[h][first + s] = (short)code;
            }
        }
        __syncthreads();
        if (m.misfit || lev + 1 >= kSubLevels || depth + lev + 1 >= kSubLevels) {
            // more nodes than particles (empty sons) or too deep: not a
            // subtree that fits here; the same decision in every thread
            if (tid == 0) {
                me.nnode = -1;
                counts->misfit = 1;
            }
            return;
        }
        for (int i = tid; i < n; i += kSubBlock) {
            const int s = m.seg[i];
            if (s == 0xffff)
                continue;
            const int c = m.kid[i >= beg[s] + m.left[s]][first + s];
            m.seg[i] = c >= 0 ? (unsigned short)(c - nfirst) : 0xffff;
        }
        ++lev;
        if (tid == 0)
            off[lev] = (unsigned short)nfirst;
        nseg = m.nnext;
        first = nfirst;
        cur ^= 1;
        __syncthreads();
    }
    for (int i = tid; i < n; i += kSubBlock) {
        w.x[0][start + i] = m.x[0][i];
        w.x[1][start + i] = m.x[1][i];
        w.x[2][start + i] = m.x[2][i];
        w.idx[start + i] = m.idx[i];
    }
    __syncthreads();
    // depth-first numbers: sizes bottom-up, ids top-down, level by level
    SubNumber &q = *reinterpret_cast<SubNumber *>(&m.x[0][0]);
    for (int l = lev - 1; l >= 0; --l) {
        const int b = off[l], e = off[l + 1];
        for (int i = b + tid; i < e; i += kSubBlock) {
            int nn = 1, nl = 0;
            for (int h = 0; h < 2; ++h) {
                const int c = m.kid[h][i];
                nn += c >= 0 ? q.nodes[c] : 0;
                nl += c >= 0 ? q.leaves[c] : 1;
            }
            q.nodes[i] = (unsigned short)nn;
            q.leaves[i] = (unsigned short)nl;
        }
        __syncthreads();
    }
    if (tid == 0) {
        q.id[0] = q.leaf0[0] = q.up[0] = 0;
        me.nnode = q.nodes[0];
        me.nleaf = q.leaves[0];
        me.nlev = lev;
    }
    __syncthreads();
    for (int l = 0; l < lev; ++l) {
        const int b = off[l], e = off[l + 1];
        for (int i = b + tid; i < e; i += kSubBlock) {
            int id = q.id[i] + 1, lf = q.leaf0[i];
            int son[2];
            for (int h = 0; h < 2; ++h) {
                const int c = m.kid[h][i];
                if (c >= 0) {
                    q.id[c] = (unsigned short)id;
                    q.leaf0[c] = (unsigned short)lf;
                    q.up[c] = (unsigned short)(i << 1 | h);
                    son[h] = id;
                    id += q.nodes[c];
                    lf += q.leaves[c];
                } else {
                    w.ld[start + lf] = m.lbeg[-c - 1] | m.llen[-c - 1] << 16;
                    son[h] = -lf - 1;
                    ++lf;
                }
            }
            w.la[start + i] = q.id[i] | q.up[i] << 12;
            w.lb[start + i] = (son[0] & 0xffff) | son[1] << 16;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------- placement
// below[s] = (nodes, leaves) in the subtree of segment s.
__global__ __launch_bounds__(kTreeBlock) void k_tree_below(TreeLevelView lv, int nseg,
                                                         const int2 *__restrict__ below_next,
                                                         const TreeSub *__restrict__ sub)
{
    const long long s = gid();
    if (s >= nseg)
        return;
    const int k[2] = {lv.kid[s].x, lv.kid[s].y};
    int nb = 1, lb = 0;
    for (int c = 0; c < 2; ++c) {
        if (k[c] >= kSubKid) {
            nb += sub[k[c] - kSubKid].nnode;
            lb += sub[k[c] - kSubKid].nleaf;
        } else if (k[c] >= 0) {
            nb += below_next[k[c]].x;
            lb += below_next[k[c]].y;
        } else {
            lb += 1;
        }
    }
    lv.below[s] = make_int2(nb, lb);
}

__device__ __forceinline__ void set_dim(float4 &v, int dir, float x)
{
    if (dir == 0)
        v.x = x;
    else if (dir == 1)
        v.y = x;
    else
        v.z = x;
}

__device__ __forceinline__ float get_dim(const float4 &v, int dir) { return dir == 0 ? v.x : dir == 1 ? v.y : v.z; }

__device__ __forceinline__ float4 box_width(const float4 &lo, const float4 &hi)
{
    return make_float4(hi.x - lo.x, hi.y - lo.y, hi.z - lo.z, 0.f);
}

__device__ __forceinline__ float4 box_center(const float4 &lo, const float4 &hi)
{
    return make_float4((float)(0.5 * (double)(hi.x + lo.x)), (float)(0.5 * (double)(hi.y + lo.y)),
                       (float)(0.5 * (double)(hi.z + lo.z)), 0.f);
}

// Leaf l, son c of a node with box [lo, hi] split at sp along dir.
__device__ __forceinline__ void place_leaf(const TreeOut &out, int l, int2 rg, int c, float4 lo, float4 hi, int dir,
                                           float sp)
{
    float4 lw = box_width(lo, hi), lc = box_center(lo, hi);
    const float lod = get_dim(lo, dir), hid = get_dim(hi, dir);
    if (c == 0) {
        set_dim(lw, dir, sp - lod);
        set_dim(lc, dir, (float)(0.5 * (double)(lod + sp)));
    } else {
        set_dim(lw, dir, hid - sp);
        set_dim(lc, dir, (float)(0.5 * (double)(hid + sp)));
    }
    out.leaf_rng[l] = rg;
    out.leaf_width[l] = lw;
    out.leaf_center[l] = lc;
}

// Depth-first ids and boxes: node s of this level has id idb[s].x, its
// subtree's leaves start at idb[s].y, its box is [lo, hi].  Writes the node,
// its leaf sons, and the ids and boxes of its node and subtree sons.
__global__ __launch_bounds__(kTreeBlock) void k_tree_place(TreeLevelView lv, int nseg, TreeLevelView nx, int dir,
                                                         TreeSub *__restrict__ sub, TreeOut out)
{
    const long long s = gid();
    if (s >= nseg)
        return;
    int id = lv.idb[s].x, lf = lv.idb[s].y;
    const float4 lo = lv.lo[s], hi = lv.hi[s];
    const int I = id;
    out.node_width[I] = box_width(lo, hi);
    out.node_center[I] = box_center(lo, hi);
    const int k[2] = {lv.kid[s].x, lv.kid[s].y};
    const float sp = lv.split[s];
    int son[2];
    ++id;
    for (int c = 0; c < 2; ++c) {
        if (k[c] < 0) {
            place_leaf(out, lf, lv.leaf[-k[c] - 1], c, lo, hi, dir, sp);
            son[c] = -lf - 1;
            ++lf;
            continue;
        }
        float4 clo = lo, chi = hi;
        set_dim(c == 0 ? chi : clo, dir, sp);
        son[c] = id;
        if (k[c] >= kSubKid) {
            TreeSub &t = sub[k[c] - kSubKid];
            t.id = id;
            t.leaf0 = lf;
            t.lo = clo;
            t.hi = chi;
            id += t.nnode;
            lf += t.nleaf;
        } else {
            nx.idb[k[c]] = make_int2(id, lf);
            nx.lo[k[c]] = clo;
            nx.hi[k[c]] = chi;
            id += nx.below[k[c]].x;
            lf += nx.below[k[c]].y;
        }
    }
    out.son[I] = make_int2(son[0], son[1]);
}

// The nodes and leaves of the subtrees, one block per subtree and one thread
// per node: its box is the root's, cut by the nearest split on the way up
// that bounds each side.
__global__ __launch_bounds__(kTreeBlock) void k_tree_place_sub(TreeScratch w, const TreeSub *__restrict__ sub,
                                                             TreeOut out)
{
    const TreeSub &t = sub[blockIdx.x];
    const int start = t.start, nnode = t.nnode;
    for (int i = threadIdx.x; i < nnode; i += kTreeBlock) {
        const unsigned a = (unsigned)w.la[start + i];
        const int lb = w.lb[start + i];
        // levels above node i in the subtree
        int lev = 0;
        for (int p = i; p > 0; p = (int)((unsigned)w.la[start + p] >> 13))
            ++lev;
        float4 lo = t.lo, hi = t.hi;
        unsigned have = 0;                           // bits 0-2: lo set, 3-5: hi set
        int p = i, dir = (t.depth + lev) % 3;
        const int mine = dir;
        while (p > 0 && have != 63u) {
            const unsigned up = (unsigned)w.la[start + p] >> 12;
            p = (int)(up >> 1);
            dir = dir == 0 ? 2 : dir - 1;
            const unsigned bit = (up & 1u) ? 1u << dir : 8u << dir;     // right son: its lower side
            if (!(have & bit)) {
                have |= bit;
                set_dim((up & 1u) ? lo : hi, dir, __int_as_float(w.lc[start + p]));
            }
        }
        const int I = t.id + (int)(a & 0xfffu);
        const float sp = __int_as_float(w.lc[start + i]);
        out.node_width[I] = box_width(lo, hi);
        out.node_center[I] = box_center(lo, hi);
        int son[2] = {(int)(short)(lb & 0xffff), lb >> 16};
        for (int c = 0; c < 2; ++c) {
            if (son[c] >= 0) {
                son[c] += t.id;
            } else {
                const int q = -son[c] - 1, r = w.ld[start + q], l = t.leaf0 + q;
                place_leaf(out, l, make_int2(start + (r & 0xffff), (int)((unsigned)r >> 16)), c, lo, hi, mine, sp);
                son[c] = -l - 1;
            }
        }
        out.son[I] = make_int2(son[0], son[1]);
    }
}

// Target marking (src/fmm.c:1226-1236): 0 when the leaf holds a particle
// with tag 1, else -1.
__global__ __launch_bounds__(kTreeBlock) void k_tree_active(const int2 *__restrict__ rng, int nleaf,
                                                          const int *__restrict__ idx, const int *__restrict__ tag,
                                                          int *__restrict__ active)
{
    const long long l = gid();
    if (l >= nleaf)
        return;
    const int2 r = rng[l];
    int a = -1;
    for (int k = 0; k < r.y; ++k)
        if (tag[idx[r.x + k]] == 1) {
            a = 0;
            break;
        }
    active[l] = a;
}

// Positions in tree order: x3 = int2pos * posi (FP64, AoS).
__global__ __launch_bounds__(kTreeBlock) void k_tree_x3(const int *__restrict__ x0, const int *__restrict__ x1,
                                                      const int *__restrict__ x2, double int2pos, long long n,
                                                      double *__restrict__ x3)
{
    const long long i = gid();
    if (i >= n)
        return;
    x3[3 * i] = int2pos * (double)x0[i];
    x3[3 * i + 1] = int2pos * (double)x1[i];
    x3[3 * i + 2] = int2pos * (double)x2[i];
}

__global__ void k_tree_root(TreeLevelView root, TreeSub *sub, float4 lo, float4 hi)
{
    if (threadIdx.x != 0)
        return;
    if (sub) {
        sub->id = sub->leaf0 = 0;
        sub->lo = lo;
        sub->hi = hi;
    } else {
        root.idb[0] = make_int2(0, 0);
        root.lo[0] = lo;
        root.hi[0] = hi;
    }
}

}  // namespace

hipError_t tree_root(const TreeLevelView *root, TreeSub *sub, float4 lo, float4 hi, hipStream_t st)
{
    k_tree_root<<<1, 64, 0, st>>>(root ? *root : TreeLevelView{}, root ? nullptr : sub, lo, hi);
    return hipGetLastError();
}

hipError_t tree_init(const int *posi, long long n, const TreeScratch &w, TreeCounts *counts, const TreeLevelView *root,
                     TreeSub *sub, hipStream_t st)
{
    k_tree_init<<<grid_of(n), kTreeBlock, 0, st>>>(posi, n, w, counts, root ? *root : TreeLevelView{},
                                                   root ? nullptr : sub);
    return hipGetLastError();
}

hipError_t tree_level(const TreeScratch &w, const TreeLevelView &lv, const TreeLevelView &nx, int level, int cap,
                      long long tiles, double int2pos, int maxleaf, int gmax, double *csum, void *units,
                      unsigned long long *mask, int *tcnt, int *tmap, TreeCounts *counts, TreeSub *sub, int subcap,
                      hipStream_t st)
{
    const int *ns = &counts->nseg[level];
    const int *x = w.x[level % 3];
    const dim3 nt = wide_grid(tiles);
    GroupUnits *u = reinterpret_cast<GroupUnits *>(units);
    k_tree_sums<<<nt, kTreeBlock, 0, st>>>(lv, ns, x, int2pos, csum, tmap);
    k_tree_units<<<nt, kUnitBlock, 0, st>>>(lv, ns, x, int2pos, csum, tmap, u);
    k_tree_mean<<<wide_grid(cap), 64, 0, st>>>(lv, ns, x, int2pos, u);
    k_tree_flags<<<nt, kTreeBlock, 0, st>>>(lv, ns, x, int2pos, mask, tcnt, tmap);
    k_tree_lists<<<nt, kTreeBlock, 0, st>>>(lv, ns, x, mask, tcnt, tmap, w.la, w.lb);
    k_tree_swap<<<nt, kTreeBlock, 0, st>>>(lv, ns, tmap, w);
    k_tree_next<<<1, kNextBlock, 0, st>>>(lv, nx, level, maxleaf, gmax, counts, sub, subcap);
    return hipGetLastError();
}

hipError_t tree_subs(const TreeScratch &w, TreeSub *sub, int nsub, double int2pos, int maxleaf, unsigned short *off,
                     TreeCounts *counts, hipStream_t st)
{
    if (nsub > 0)
        k_tree_sub<<<wide_grid(nsub), kSubBlock, 0, st>>>(w, sub, nsub, int2pos, maxleaf, off, counts);
    return hipGetLastError();
}

hipError_t tree_below(const TreeLevelView &lv, int nseg, const int2 *below_next, const TreeSub *sub, hipStream_t st)
{
    k_tree_below<<<grid_of(nseg), kTreeBlock, 0, st>>>(lv, nseg, below_next, sub);
    return hipGetLastError();
}

hipError_t tree_place(const TreeLevelView &lv, int nseg, const TreeLevelView &nx, int dir, TreeSub *sub,
                      const TreeOut &out, hipStream_t st)
{
    k_tree_place<<<grid_of(nseg), kTreeBlock, 0, st>>>(lv, nseg, nx, dir, sub, out);
    return hipGetLastError();
}

hipError_t tree_place_subs(const TreeScratch &w, const TreeSub *sub, int nsub, const TreeOut &out, hipStream_t st)
{
    if (nsub > 0)
        k_tree_place_sub<<<(unsigned)nsub, kTreeBlock, 0, st>>>(w, sub, out);
    return hipGetLastError();
}

hipError_t tree_finish(const TreeScratch &w, const TreeOut &out, int nleaf, const int *tag, double int2pos,
                       long long n, double *x3, hipStream_t st)
{
    k_tree_active<<<grid_of(nleaf), kTreeBlock, 0, st>>>(out.leaf_rng, nleaf, w.idx, tag, out.leaf_active);
    k_tree_x3<<<grid_of(n), kTreeBlock, 0, st>>>(w.x[0], w.x[1], w.x[2], int2pos, n, x3);
    return hipGetLastError();
}

}  // namespace pp2p
