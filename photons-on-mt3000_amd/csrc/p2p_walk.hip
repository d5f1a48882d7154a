// Interaction lists on the device: the symmetric dual walk of the kd-tree
// (walk_task_p2p, src/fmm.c:656-792, with the acceptance test of
// src/fmm.c:411-479) run level-synchronously instead of recursively.
//
// A frame is a (target, source) pair of tree cells; >= 0 names a node,
// < 0 a leaf as -(id + 1).  The recursive walk calls, from a frame:
//   node self pair   -> (s0,s0) (s0,s1) (s1,s0) (s1,s1)
//   leaf-node pair   -> opened (accept == 0): the node's two sons, else nothing
//   node-node pair   -> opened: the two sons of the wider box (sum of widths)
//   leaf-leaf pair   -> emits the task when the target leaf holds a local
//                       particle (active >= 0)
// Round r holds the opened frames at call depth r in depth-first order; what
// becomes of a frame's children (opened, task, well separated, nothing) is
// decided with the frame, so a child that is not opened is never stored: half of
// all pairs are leaf pairs, another eighth is dropped.  Three passes turn
// the rounds into the task list in the order the recursive walk emits it:
//   forward   codes of the children, and the opened ones placed as round
//             r + 1 by a prefix sum over the round within the same launch (the
//             decoupled look-back of Merrill and Garland)
//   backward  tasks below each frame: its own plus its opened children's, which
//             lie next to each other
//   positions each frame's first task position, handed from parent to child;
//             the frames write their tasks there
// The rounds' sizes stay on the device; the host reads them once per group of
// rounds.  Bound by HBM in the large rounds (about 70 bytes per opened frame in
// all, and 160 bytes of cells from L2) and by launches and a chain of five
// dependent loads in the small ones.  256^3 clustered tree (1.0 10^8 opened
// frames of 2.1 10^8 pairs, 8.7 10^7 tasks): 4.8 ms a call, where storing every
// pair as a frame, with separate kernels for codes, library scans and children
// and a host wait per round, took 10.7 ms; 64^3 2.15 -> 0.68 ms, 16^3 1.46 ->
// 0.29 ms.
// The geometry is FP32 with each operation rounded on its own (no
// contraction), as the host's cpuType arithmetic.
#include "p2p_walk.h"

#pragma clang fp contract(off)

namespace pp2p {
namespace {

constexpr int kWalkBlock = 256;
static_assert(kWalkBlock == kWalkTile, "a thread per frame in the small tiles");
constexpr int kWalkWaves = kWalkBlock / 64;
constexpr int kPerThread = 4;

// 1: well separated (multipole), 0: open, -1: beyond the cutoff.  Operation
// order and types as src/fmm.c:411-479: the half-sum of widths in FP64, the
// distance test on the gap vector, the opening test on the centre distance.
__device__ __forceinline__ int accept(const float4 wi, const float4 wj, float dx, float dy, float dz,
                                      float open_angle, float cutoff)
{
    const float w0 = (float)((double)(wi.x + wj.x) * 0.5);
    const float w1 = (float)((double)(wi.y + wj.y) * 0.5);
    const float w2 = (float)((double)(wi.z + wj.z) * 0.5);
    float m0 = dx < 0.0f ? -dx : dx;
    float m1 = dy < 0.0f ? -dy : dy;
    float m2 = dz < 0.0f ? -dz : dz;
    m0 -= w0;
    m1 -= w1;
    m2 -= w2;
    if (m0 <= 0.0f)
        m0 = 0.0f;
    if (m1 <= 0.0f)
        m1 = 0.0f;
    if (m2 <= 0.0f)
        m2 = 0.0f;
    const float dd2 = dx * dx + dy * dy + dz * dz;
    if ((double)(m0 + m1 + m2) < 1.0e-15)
        return 0;
    const float dm2 = m0 * m0 + m1 * m1 + m2 * m2;
    if (dm2 > cutoff * cutoff)
        return -1;
    float wmax = w0;
    if (w1 > wmax)
        wmax = w1;
    if (w2 > wmax)
        wmax = w2;
    wmax = fabsf(wmax);
    wmax *= 2.0f;
    return (wmax * wmax < open_angle * open_angle * dd2) ? 1 : 0;
}

__device__ __forceinline__ WalkCell cell_at(const WalkCell *cells, int nnode, int id)
{
    return cells[id >= 0 ? id : nnode - id - 1];
}

__global__ __launch_bounds__(kWalkBlock) void k_walk_cells(WalkTree t, WalkCell *__restrict__ cells)
{
    const int i = blockIdx.x * kWalkBlock + threadIdx.x;
    if (i >= t.nnode + t.nleaf)
        return;
    const bool node = i < t.nnode;
    const int l = i - t.nnode;
    const float4 c = node ? t.node_center[i] : t.leaf_center[l];
    const float4 w = node ? t.node_width[i] : t.leaf_width[l];
    const int2 s = node ? t.son[i] : make_int2(t.leaf_active[l], 0);
    cells[i] = WalkCell{c.x, c.y, c.z, s.x, w.x, w.y, w.z, s.y};
}

__global__ __launch_bounds__(kWalkBlock) void k_walk_begin(WalkFrames w, WalkRound *__restrict__ rounds, int count,
                                                         WalkRound cur)
{
    const long long i = (long long)blockIdx.x * kWalkBlock + threadIdx.x;
    const long long step = (long long)gridDim.x * kWalkBlock;
    for (long long k = i; k < count; k += step) {
        WalkRound r{};
        if (k == 0) {
            r.n = cur.n;
            r.fbase = cur.fbase;
            r.tbase = cur.tbase;
        }
        rounds[k] = r;
    }
    if (i == 0 && cur.fbase == 0)
        w.f[0] = make_int2(0, 0);
    for (long long k = cur.tbase + i; k < w.tcap; k += step)
        w.look[k] = 0ull;
}

// What becomes of the child pair (i, j), not the same node: `active` is the
// target leaf's mark, acc the acceptance of the two cells (symmetric in them: the
// half-sum of widths, squares and magnitudes of the distance).
__device__ __forceinline__ unsigned child_code(int i, int j, int active, int acc)
{
    if (i < 0 && j < 0)
        return active >= 0 ? 2u : 0u;
    return acc == 0 ? 1u : acc == 1 ? 3u : 0u;
}

__device__ __forceinline__ int accept_cells(const WalkCell &a, const WalkCell &b, float open_angle, float cutoff)
{
    return accept(make_float4(a.wx, a.wy, a.wz, 0.f), make_float4(b.wx, b.wy, b.wz, 0.f), a.cx - b.cx, a.cy - b.cy,
                  a.cz - b.cz, open_angle, cutoff);
}

__device__ __forceinline__ unsigned opened(unsigned code)      // children with code 1
{
    return __popc(code & ~(code >> 1) & 0x55u);
}
__device__ __forceinline__ unsigned tasks(unsigned code) { return __popc((code >> 1) & ~code & 0x55u); }
__device__ __forceinline__ unsigned separated(unsigned code) { return __popc(code & (code >> 1) & 0x55u); }

// the children codes of a stored code: bit 4 of a two-child frame is no code
__device__ __forceinline__ unsigned child_bits(int2 f, unsigned code) { return f.x == f.y ? code : code & 15u; }

// child h of frame f; (sx, sy): the sons of the split cell
__device__ __forceinline__ int2 child_of(int2 f, unsigned code, int sx, int sy, int h)
{
    if (f.x == f.y)
        return make_int2(h & 2 ? sy : sx, h & 1 ? sy : sx);
    const int s = h ? sy : sx;
    return code & 16u ? make_int2(s, f.y) : make_int2(f.x, s);
}

// exclusive prefix and total of small counts (0..4) over the wave
__device__ __forceinline__ unsigned wave_count(unsigned c, unsigned long long below, unsigned &total)
{
    const unsigned long long b0 = __ballot(c & 1u), b1 = __ballot(c & 2u), b2 = __ballot(c & 4u);
    total = __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
    return __popcll(b0 & below) + 2 * __popcll(b1 & below) + 4 * __popcll(b2 & below);
}

constexpr unsigned long long kLookSum = 1ull << 62, kLookAll = 2ull << 62, kLookValue = kLookSum - 1;

// Frames per thread of a round's tiles: four in the large rounds (fewer
// tickets and look-backs per frame), one up to 2^18 frames, which would not
// fill the chip otherwise (64^3 walk, all rounds at four: 1.04 ms; 0.68 so).
__host__ __device__ constexpr int walk_per(unsigned n) { return n <= (unsigned)kWalkSmall * kWalkTile ? 1 : kPerThread; }

struct OpenShared {
    unsigned open[kWalkWaves], sep[kWalkWaves];
    unsigned long long before;
};

// One tile of the forward pass; the thread's tasks are returned.  No branch
// between the loads of a thread's frames, so that they are in flight together:
// frame, its two cells, the split one's sons.
template <int PER>
__device__ __forceinline__ unsigned open_tile(const WalkCell *__restrict__ cells, int nnode, float open_angle,
                                              float cutoff, const WalkFrames &w, WalkRound *round, unsigned tile,
                                              unsigned n, unsigned ntile, long long fbase, unsigned long long *look,
                                              int *sep, OpenShared &sh)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    const long long next = fbase + n;
    auto at_of = [&](int u) { return tile * (unsigned)(PER * kWalkBlock) + (unsigned)((wave * PER + u) * 64 + lane); };
    int2 f[PER];
    int sx[PER], sy[PER];
    unsigned code[PER], at[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u)
        f[u] = w.f[fbase + min(at_of(u), n - 1)];
    unsigned wopen = 0, wsep = 0, ntask = 0;
    constexpr int kTwo = PER < 2 ? 1 : 2;
#pragma unroll
    for (int v = 0; v < PER; v += kTwo) {
        WalkCell other[kTwo], p[kTwo], q[kTwo];
        bool self[kTwo], ta[kTwo];
#pragma unroll
        for (int h = 0; h < kTwo; ++h) {
            p[h] = cell_at(cells, nnode, f[v + h].x);
            q[h] = cell_at(cells, nnode, f[v + h].y);
        }
#pragma unroll
        for (int h = 0; h < kTwo; ++h) {
            const int2 g = f[v + h];
            // which cell is split: the target's if it is a node and the
            // source's a leaf or narrower (sum of widths)
            self[h] = g.x == g.y;
            ta[h] = self[h] || (g.x >= 0 && (g.y < 0 || p[h].wx + p[h].wy + p[h].wz > q[h].wx + q[h].wy + q[h].wz));
            sx[v + h] = ta[h] ? p[h].a : q[h].a;
            sy[v + h] = ta[h] ? p[h].b : q[h].b;
            other[h] = ta[h] ? q[h] : p[h];
        }
#pragma unroll
        for (int h = 0; h < kTwo; ++h) {
            p[h] = cell_at(cells, nnode, sx[v + h]);
            q[h] = cell_at(cells, nnode, sy[v + h]);
        }
#pragma unroll
        for (int h = 0; h < kTwo; ++h) {
            const int u = v + h, x = sx[u], y = sy[u];
            const int ap = accept_cells(p[h], self[h] ? q[h] : other[h], open_angle, cutoff);
            const int aq = accept_cells(q[h], other[h], open_angle, cutoff);
            unsigned c;
            if (self[h])
                c = (x < 0 ? child_code(x, x, p[h].a, 0) : 1u) | child_code(x, y, p[h].a, ap) << 2 |
                    child_code(y, x, q[h].a, ap) << 4 | (y < 0 ? child_code(y, y, q[h].a, 0) : 1u) << 6;
            else if (ta[h])
                c = 16u | child_code(x, f[u].y, p[h].a, ap) | child_code(y, f[u].y, q[h].a, aq) << 2;
            else
                c = child_code(f[u].x, x, other[h].a, ap) | child_code(f[u].x, y, other[h].a, aq) << 2;
            const bool in = at_of(u) < n;
            code[u] = c;
            if (in)
                w.code[fbase + at_of(u)] = (unsigned char)c;
            const unsigned bits = in ? child_bits(f[u], c) : 0u;
            unsigned t;
            at[u] = wopen + wave_count(opened(bits), below, t);
            wopen += t;
            wave_count(separated(bits), below, t);
            wsep += t;
            ntask += tasks(bits);
        }
    }
    if (lane == 0) {
        sh.open[wave] = wopen;
        sh.sep[wave] = wsep;
    }
    __syncthreads();
    unsigned bopen = 0, bsep = 0, mine = 0;
#pragma unroll
    for (int q = 0; q < kWalkWaves; ++q) {
        mine += q < wave ? sh.open[q] : 0;
        bopen += sh.open[q];
        bsep += sh.sep[q];
    }
    if (wave == 0) {
        const unsigned long long sum = bopen | (unsigned long long)bsep << 31;
        unsigned long long before = 0;
        if (lane == 0)
            __hip_atomic_store(&look[tile], (tile ? kLookSum : kLookAll) | sum, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        for (int last = (int)tile - 1; last >= 0; last -= 64) {
            unsigned long long v;
            do {
                v = last - lane >= 0 ? __hip_atomic_load(&look[last - lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                     : kLookAll;
            } while (__ballot(v < kLookSum));
            const unsigned long long all = __ballot(v >= kLookAll);
            const int upto = all ? __builtin_ctzll(all) : 63;
            unsigned long long t = lane <= upto ? v & kLookValue : 0ull;
            for (int o = 32; o > 0; o >>= 1)
                t += __shfl_xor(t, o, 64);
            before += t;
            if (all)
                break;
        }
        if (lane == 0) {
            if (tile)
                __hip_atomic_store(&look[tile], kLookAll | (before + sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sh.before = before;
            sep[tile] = (int)(before >> 31);
            if (tile == ntile - 1) {
                const unsigned long long t = before + sum;
                const unsigned nn = (unsigned)(t & 0x7fffffffull);
                round->nsep = (unsigned)(t >> 31);
                round[1].n = nn;
                round[1].fbase = next;
                round[1].tbase = round->tbase + ntile;
                round[1].over = next + nn > w.cap;
            }
        }
    }
    __syncthreads();
    const unsigned base = (unsigned)(sh.before & 0x7fffffffull) + mine;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const unsigned i = at_of(u);
        if (i >= n)
            continue;
        unsigned o = base + at[u];
        w.off[fbase + i] = o;
        const unsigned bits = child_bits(f[u], code[u]);
#pragma unroll
        for (int h = 0; h < 4; ++h)
            if (((bits >> (2 * h)) & 3u) == 1u) {
                if (next + o < w.cap)
                    w.f[next + o] = child_of(f[u], code[u], sx[u], sy[u], h);
                ++o;
            }
    }
    return ntask;
}

// Forward.  A block takes tiles in order from the round's ticket, so every
// tile waits only for tiles that are already running; tile words carry
// (opened | separated << 31) and whether they hold the tile's sum or the sum up to
// and with it.
__global__ __launch_bounds__(kWalkBlock) void k_walk_open(const WalkCell *__restrict__ cells, int nnode,
                                                        float open_angle, float cutoff, WalkFrames w,
                                                        WalkRound *round)
{
    __shared__ unsigned s_tile;
    __shared__ OpenShared sh;
    __shared__ unsigned long long s_task[kWalkWaves];
    const unsigned n = round->n;
    if (n == 0 || round->over)
        return;
    const int per = walk_per(n);
    const unsigned ntile = (n + per * kWalkBlock - 1) / (per * kWalkBlock);
    if (blockIdx.x >= ntile)
        return;                                      // every ticket is an atomic on one address
    const long long fbase = round->fbase;
    unsigned long long *look = w.look + round->tbase;
    int *sep = w.sep + round->tbase;
    unsigned long long ntask = 0;
    for (;;) {
        if (threadIdx.x == 0)
            s_tile = atomicAdd(&round->ticket, 1u);
        __syncthreads();
        const unsigned tile = s_tile;
        if (tile >= ntile)
            break;
        ntask += per == 1 ? open_tile<1>(cells, nnode, open_angle, cutoff, w, round, tile, n, ntile, fbase, look, sep, sh)
                          : open_tile<kPerThread>(cells, nnode, open_angle, cutoff, w, round, tile, n, ntile, fbase,
                                                  look, sep, sh);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = 32; o > 0; o >>= 1)
        ntask += __shfl_xor(ntask, o, 64);
    if (lane == 0)
        s_task[wave] = ntask;
    __syncthreads();
    if (threadIdx.x == 0) {
        ntask = 0;
        for (int q = 0; q < kWalkWaves; ++q)
            ntask += s_task[q];
        if (ntask)
            atomicAdd(&round->ntask, ntask);
    }
}

// Backward: tasks at and below each frame.
__global__ __launch_bounds__(kWalkBlock) void k_walk_below(WalkFrames w, long long fbase, unsigned n)
{
    const unsigned i = blockIdx.x * kWalkBlock + threadIdx.x;
    if (i >= n)
        return;
    const unsigned bits = child_bits(w.f[fbase + i], w.code[fbase + i]);
    const unsigned k = opened(bits);
    int v = (int)tasks(bits);
    const int *c = w.cnt + fbase + n + w.off[fbase + i];
    for (unsigned j = 0; j < k; ++j)
        v += c[j];
    w.cnt[fbase + i] = v;
}

// Positions: cnt holds the frame's first task position; an opened child's
// count is replaced by its position.
template <bool SEP, int PER>
__global__ __launch_bounds__(kWalkBlock) void k_walk_emit(const WalkCell *__restrict__ cells, int nnode, int nleaf,
                                                        WalkFrames w, long long fbase, long long tbase, unsigned n,
                                                        int *__restrict__ task_t, int *__restrict__ task_s,
                                                        int *__restrict__ ct, int *__restrict__ cs)
{
    __shared__ unsigned s_sep[kWalkWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned code[PER], rank[PER];
    int2 f[PER];
    unsigned wsep = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const unsigned i = blockIdx.x * (unsigned)(PER * kWalkBlock) + (wave * PER + u) * 64 + lane;
        code[u] = i < n ? w.code[fbase + i] : 0;
        f[u] = i < n ? w.f[fbase + i] : make_int2(0, 0);
        if (SEP) {
            unsigned t;
            rank[u] = wsep + wave_count(separated(child_bits(f[u], code[u])), below, t);
            wsep += t;
        }
    }
    unsigned sbase = 0;
    if (SEP) {
        if (lane == 0)
            s_sep[wave] = wsep;
        __syncthreads();
        sbase = (unsigned)w.sep[tbase + blockIdx.x];
        for (int q = 0; q < wave; ++q)
            sbase += s_sep[q];
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const unsigned i = blockIdx.x * (unsigned)(PER * kWalkBlock) + (wave * PER + u) * 64 + lane;
        if (i >= n)
            continue;
        const unsigned bits = child_bits(f[u], code[u]);
        int p = w.cnt[fbase + i];
        int *c = w.cnt + fbase + n + w.off[fbase + i];
        unsigned r = SEP ? sbase + rank[u] : 0;
        int sx = 0, sy = 0;
        if (tasks(bits) || (SEP && separated(bits))) {
            const bool own = f[u].x == f[u].y || (code[u] & 16u);
            const int s = own ? f[u].x : f[u].y;     // the split cell is a node
            sx = cells[s].a;
            sy = cells[s].b;
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const unsigned k = (bits >> (2 * h)) & 3u;
            if (k == 1u) {
                const int below_child = *c;
                *c++ = p;
                p += below_child;
            } else if (k == 2u) {
                const int2 q = child_of(f[u], code[u], sx, sy, h);
                task_t[p] = -q.x - 1;
                task_s[p] = -q.y - 1;
                ++p;
            } else if (SEP && k == 3u) {
                const int2 q = child_of(f[u], code[u], sx, sy, h);
                ct[r] = q.x < 0 ? -q.x - 1 : nleaf + q.x;
                cs[r] = q.y < 0 ? -q.y - 1 : nleaf + q.y;
                ++r;
            }
        }
    }
}

inline unsigned grid_of(long long n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

hipError_t walk_cells(const WalkTree &t, WalkCell *cells, hipStream_t st)
{
    k_walk_cells<<<grid_of((long long)t.nnode + t.nleaf, kWalkBlock), kWalkBlock, 0, st>>>(t, cells);
    return hipGetLastError();
}

hipError_t walk_begin(const WalkFrames &w, WalkRound *rounds, int count, const WalkRound &cur, hipStream_t st)
{
    const long long k = w.tcap - cur.tbase > count ? w.tcap - cur.tbase : count;
    const unsigned g = grid_of(k, kWalkBlock);
    k_walk_begin<<<g < 1024 ? g : 1024, kWalkBlock, 0, st>>>(w, rounds, count, cur);
    return hipGetLastError();
}

hipError_t walk_open(const WalkTree &t, const WalkCell *cells, const WalkFrames &w, WalkRound *round, int blocks,
                     hipStream_t st)
{
    k_walk_open<<<(unsigned)blocks, kWalkBlock, 0, st>>>(cells, t.nnode, t.open_angle, t.cutoff, w, round);
    return hipGetLastError();
}

hipError_t walk_below(const WalkFrames &w, long long fbase, unsigned n, hipStream_t st)
{
    k_walk_below<<<grid_of(n, kWalkBlock), kWalkBlock, 0, st>>>(w, fbase, n);
    return hipGetLastError();
}

hipError_t walk_emit(const WalkTree &t, const WalkCell *cells, const WalkFrames &w, long long fbase, long long tbase,
                     unsigned n, unsigned nsep, int *task_t, int *task_s, int *ct, int *cs, hipStream_t st)
{
    const int per = walk_per(n);
    const unsigned g = grid_of(n, per * kWalkBlock);
    auto run = [&](auto kernel) {
        kernel<<<g, kWalkBlock, 0, st>>>(cells, t.nnode, t.nleaf, w, fbase, tbase, n, task_t, task_s, ct, cs);
    };
    if (per == 1)
        nsep ? run(k_walk_emit<true, 1>) : run(k_walk_emit<false, 1>);
    else
        nsep ? run(k_walk_emit<true, kPerThread>) : run(k_walk_emit<false, kPerThread>);
    return hipGetLastError();
}

}  // namespace pp2p
