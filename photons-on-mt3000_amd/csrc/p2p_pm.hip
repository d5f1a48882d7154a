// Particle-mesh long-range force (partmesh_kick, src/partmesh.c:1476-2954, and
// its convolution, src/conv.f90:168-352) with the whole periodic mesh on one GPU.
//
// * CIC weights in the reference's FP32 arithmetic: posf = (float)(posi *
//   INT2POS); i = (int)(posf * norm); w = (posf - (i + 0.5) delta) norm with the
//   neighbour on the side of w (src/partmesh.c:1569-1612).
// * The deposit adds the FP32 products MASSPART * wx * wy * wz into an FP64
//   mesh with atomics, first summed per chunk of particles in LDS (the
//   reference sums in FP32 in particle order).
// * The Green's function multiplies the FP64 r2c spectrum in place; it
//   includes the reference's conversion of mass per cell to density.
// * The acceleration: 4-point central differences of the potential at the 8
//   CIC cells, weighted by the CIC weights, in FP64; stored as FP32 like the
//   reference's acc arrays.
// Cell indices wrap modulo N where the reference reads its ghost layers.
#include "p2p_pm.h"

#pragma clang fp contract(off)

namespace pp2p {
namespace {

constexpr int kPmBlock = 256;
// conv.f90's M_PI = 3.1415926, a REAL(cputype) constant
constexpr double kPiRef = (double)3.1415926f;

struct Axis {
    int i, ii;
    float w, wn;     // weight of the neighbour ii, of the own cell i
};

__device__ __forceinline__ Axis cic_axis(float posf, float norm, float delta)
{
    Axis a;
    a.i = (int)(posf * norm);
    float w = (float)(((double)posf - ((double)a.i + 0.5) * (double)delta) * (double)norm);
    if (w > 0.0f) {
        a.ii = a.i + 1;
    } else {
        w = -w;
        a.ii = a.i - 1;
    }
    a.w = w;
    a.wn = (float)(1.0 - (double)w);
    return a;
}

__device__ __forceinline__ int wrap(int i, int n)
{
    int r = i % n;
    return r < 0 ? r + n : r;
}

// cells per length, and a cell's length, as the reference rounds them
struct Grid {
    float norm, delta;
};

inline Grid grid_of(const PmArgs &a)
{
    const float norm = (float)a.nside / a.box;
    return Grid{norm, (float)(1.0 / (double)norm)};
}

__device__ __forceinline__ void particle_axes(const PmArgs &a, const Grid &g, long long p, Axis ax[3])
{
    const int *pc[3] = {a.px, a.py, a.pz};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float posf = (float)((double)pc[d][p * a.stride] * a.int2pos);
        ax[d] = cic_axis(posf, g.norm, g.delta);
    }
}

// One block deposits a chunk of kPmChunk consecutive particles.  Particles
// that arrive in spatial order (tree order) cover few cells per chunk: the
// chunk's cells (unwrapped indices, both CIC neighbours) are bounded first,
// and when the box fits in kPmTile cells the chunk sums into LDS and adds each
// touched cell to the mesh once.  Otherwise the tile is a hash table of the
// touched cells; a corner that finds no place within kPmProbes goes to the mesh.
// Neighbouring particles share cells, and LDS adds to one address take turns; so
// the tile holds as many copies of the box as fit (a power of two, kPmCopies at
// most) and lane l adds to copy l mod their number.  Bound by the adds to the
// mesh, 3 10^10 a second: with one copy and every corner of a chunk that does not
// fit sent there, 1.7 10^7 particles in tree order (256^3 mesh, clustered) took
// 1850 us, now 960; 3.6 10^5 of 64^3 70, now 38; 10^6 in no order 490, now 390.
constexpr int kPmChunk = 1024;
constexpr int kPmTile = 4096;
constexpr int kPmProbes = 8;
constexpr int kPmCopies = 64;
constexpr int kPmOwn = kPmChunk / kPmBlock;          // particles per thread

__device__ __forceinline__ bool is_local(const PmArgs &a, long long p)
{
    return !a.tag || a.tag[a.tag_idx ? a.tag_idx[p] : p] == 1;
}

__device__ __forceinline__ bool local_particle(const PmArgs &a, long long p)
{
    return p < a.n && is_local(a, p);
}

__device__ __forceinline__ void hash_add(int *key, double *tile, double *rho, int cell, double m)
{
    unsigned h = (unsigned)cell * 2654435761u >> 20;
    static_assert(kPmTile == 1 << 12, "bits of the hash");
    for (int q = 0; q < kPmProbes; ++q) {
        int k = __hip_atomic_load(&key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k < 0)
            k = atomicCAS(&key[h], -1, cell);
        if (k < 0 || k == cell) {
            atomicAdd(&tile[h], m);
            return;
        }
        h = (h + 1) & (kPmTile - 1);
    }
    atomicAdd(&rho[cell], m);
}

__global__ __launch_bounds__(kPmBlock) void k_pm_deposit(PmArgs a, Grid g, double *__restrict__ rho)
{
    __shared__ double tile[kPmTile];
    __shared__ int key[kPmTile];                  // hash table: the mesh cell, -1: free
    __shared__ int lo[3], hi[3];
    const int N = a.nside;
    const long long p0 = (long long)blockIdx.x * kPmChunk;
    if (threadIdx.x < 3) {
        lo[threadIdx.x] = 0x7fffffff;
        hi[threadIdx.x] = -0x7fffffff;
    }
    __syncthreads();
    Axis ax[kPmOwn][3];
    bool mine[kPmOwn];
    int l[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, h[3] = {-0x7fffffff, -0x7fffffff, -0x7fffffff};
#pragma unroll
    for (int u = 0; u < kPmOwn; ++u) {
        const long long p = p0 + u * kPmBlock + threadIdx.x;
        mine[u] = local_particle(a, p);
        particle_axes(a, g, p < a.n ? p : a.n - 1, ax[u]);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (mine[u]) {
                l[d] = min(l[d], min(ax[u][d].i, ax[u][d].ii));
                h[d] = max(h[d], max(ax[u][d].i, ax[u][d].ii));
            }
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        atomicMin(&lo[d], l[d]);
        atomicMax(&hi[d], h[d]);
    }
    __syncthreads();
    if (hi[0] < lo[0])
        return;                                   // no local particle in the chunk
    // (indices of particles far outside the box end at the integers' range)
    const long long ex = (long long)hi[0] - lo[0], ey = (long long)hi[1] - lo[1], ez = (long long)hi[2] - lo[2];
    const bool fits = ex < kPmTile && ey < kPmTile && ez < kPmTile && (ex + 1) * (ey + 1) * (ez + 1) <= kPmTile;
    const int sx = fits ? (int)ex + 1 : 1, sy = fits ? (int)ey + 1 : 1, sz = fits ? (int)ez + 1 : 1;
    const int ncell = sx * sy * sz;
    int lg = 0;                                   // log2 of the copies
    if (fits) {
        while ((2 << lg) <= kPmCopies && (ncell << (lg + 1)) <= kPmTile)
            ++lg;
        for (int c = threadIdx.x; c < ncell << lg; c += kPmBlock)
            tile[c] = 0.0;
    } else {
        for (int c = threadIdx.x; c < kPmTile; c += kPmBlock) {
            tile[c] = 0.0;
            key[c] = -1;
        }
    }
    __syncthreads();
    const int copy = threadIdx.x & ((1 << lg) - 1);
#pragma unroll
    for (int u = 0; u < kPmOwn; ++u) {
        if (!mine[u])
            continue;
        const Axis &X = ax[u][0], &Y = ax[u][1], &Z = ax[u][2];
        const int cx[2] = {X.i, X.ii}, cy[2] = {Y.i, Y.ii}, cz[2] = {Z.i, Z.ii};
        const float wx[2] = {X.wn, X.w}, wy[2] = {Y.wn, Y.w}, wz[2] = {Z.wn, Z.w};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int x = c & 1, y = (c >> 1) & 1, z = c >> 2;
            const float m = ((a.mass * wx[x]) * wy[y]) * wz[z];
            if (fits)
                atomicAdd(&tile[((((cx[x] - lo[0]) * sy + (cy[y] - lo[1])) * sz + (cz[z] - lo[2])) << lg) + copy],
                          (double)m);
            else
                hash_add(key, tile, rho, (wrap(cx[x], N) * N + wrap(cy[y], N)) * N + wrap(cz[z], N), (double)m);
        }
    }
    __syncthreads();
    if (!fits) {
        for (int c = threadIdx.x; c < kPmTile; c += kPmBlock)
            if (key[c] >= 0)
                atomicAdd(&rho[key[c]], tile[c]);
        return;
    }
    for (int c = threadIdx.x; c < ncell; c += kPmBlock) {
        double v = 0.0;
        for (int k = 0; k < 1 << lg; ++k)         // each lane from another copy on: other banks
            v += tile[(c << lg) + ((k + c) & ((1 << lg) - 1))];
        if (v == 0.0)
            continue;
        const int x = c / (sy * sz), y = (c / sz) % sy, z = c % sz;
        atomicAdd(&rho[((long long)wrap(lo[0] + x, N) * N + wrap(lo[1] + y, N)) * N + wrap(lo[2] + z, N)], v);
    }
}

__device__ __forceinline__ double sinc_ref(int n, int N)
{
    if (n == 0)
        return 1.0;
    const double x = kPiRef * (double)n / (double)N;
    return sin(x) / x;
}

// spectrum [N][N][N/2+1]: x (l) slowest, the halved axis z (n) fastest
__global__ __launch_bounds__(kPmBlock) void k_pm_green(int N, double ismth2, double pref, double2 *__restrict__ spec)
{
    const int nh = N / 2 + 1;
    const long long e = (long long)blockIdx.x * kPmBlock + threadIdx.x;
    const long long total = (long long)N * N * nh;
    if (e >= total)
        return;
    const int n = (int)(e % nh);
    const int m0 = (int)((e / nh) % N);
    const int l0 = (int)(e / ((long long)nh * N));
    const int l = l0 > N / 2 ? l0 - N : l0;
    const int m = m0 > N / 2 ? m0 - N : m0;
    double g = 0.0;
    if (l != 0 || m != 0 || n != 0) {
        const double k2 = (double)(l * l + m * m + n * n);
        const double ff = 1.0 / (sinc_ref(l, N) * sinc_ref(m, N) * sinc_ref(n, N));
        const double ff2 = ff * ff;
        g = exp(-k2 * ismth2) / k2 * (ff2 * ff2) * pref;
    }
    double2 v = spec[e];
    v.x *= g;
    v.y *= g;
    spec[e] = v;
}

// grad[cell][d] = f1 invx (p[+1] - p[-1]) - f2 invx (p[+2] - p[-2]) along d:
// the reference evaluates this difference at each of a particle's 8 CIC
// cells (src/partmesh.c:2694-2922); it depends on the cell alone.  Rows of
// N + 1 cells, the last a copy of the first: the two cells that the
// interpolation reads along z are 48 consecutive bytes, three wide loads in
// place of six.  With three planes the interpolation of 1.7 10^7 particles in tree
// order took 990 us, now 660 (bound by the gathers); of 10^6 in any order 97, now 44.
constexpr int kGradZ = 64, kGradY = kPmBlock / kGradZ;

__global__ __launch_bounds__(kPmBlock) void k_pm_gradient(const double *__restrict__ pot, int N, double invx,
                                                          double *__restrict__ grad)
{
    const int z = blockIdx.x * kGradZ + threadIdx.x, y = blockIdx.y * kGradY + threadIdx.y, x = blockIdx.z;
    if (z >= N || y >= N)
        return;
    const double f1 = (double)(float)(4.0 / 3.0), f2 = (double)(float)(1.0 / 6.0);
    double g[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        auto at = [&](int o) {
            int r[3] = {x, y, z};
            r[d] += o;
            r[d] += r[d] < 0 ? N : r[d] >= N ? -N : 0;
            return pot[((long long)r[0] * N + r[1]) * N + r[2]];
        };
        g[d] = f1 * invx * (at(1) - at(-1)) - f2 * invx * (at(2) - at(-2));
    }
    double *row = grad + ((long long)x * N + y) * (N + 1) * 3;
#pragma unroll
    for (int d = 0; d < 3; ++d)
        row[z * 3 + d] = g[d];
    if (z == 0)
        for (int d = 0; d < 3; ++d)
            row[N * 3 + d] = g[d];
}

// acc[d][p] = sum over the 8 CIC cells of wx wy wz grad[cell][d], in the
// reference's corner order
__global__ __launch_bounds__(kPmBlock) void k_pm_interp(PmArgs a, Grid g, const double *__restrict__ grad,
                                                        float *__restrict__ acc, double *__restrict__ acc64)
{
    const long long p = (long long)blockIdx.x * kPmBlock + threadIdx.x;
    if (p >= a.n)
        return;
    if (!is_local(a, p)) {
        if (acc) {
            acc[p] = 0.0f;
            acc[a.n + p] = 0.0f;
            acc[2 * a.n + p] = 0.0f;
        }
        return;
    }
    Axis ax[3];
    particle_axes(a, g, p, ax);
    const int N = a.nside;
    const int cx[2] = {wrap(ax[0].i, N), wrap(ax[0].ii, N)};
    const int cy[2] = {wrap(ax[1].i, N), wrap(ax[1].ii, N)};
    const int z0 = wrap(min(ax[2].i, ax[2].ii), N);
    const bool below = ax[2].ii < ax[2].i;           // the z neighbour comes first
    const double wx[2] = {ax[0].wn, ax[0].w}, wy[2] = {ax[1].wn, ax[1].w}, wz[2] = {ax[2].wn, ax[2].w};
    struct Pair {
        double v[2][3];
    } r[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        __builtin_memcpy(&r[c], grad + (((long long)cx[c & 1] * N + cy[c >> 1]) * (N + 1) + z0) * 3, sizeof(Pair));
    double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int x = c & 1, y = (c >> 1) & 1, z = c >> 2;
        const double w = wx[x] * wy[y] * wz[z];
#pragma unroll
        for (int d = 0; d < 3; ++d)
            s[d] += w * (below ? r[c & 3].v[1 - z][d] : r[c & 3].v[z][d]);
    }
    if (acc) {
        for (int d = 0; d < 3; ++d)
            acc[d * a.n + p] = (float)s[d];
    } else {
        for (int d = 0; d < 3; ++d)
            acc64[d * a.n + p] += s[d];
    }
}

__global__ void k_pm_zero(double *p, long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        p[i] = 0.0;
}

inline unsigned blocks_of(long long n) { return (unsigned)((n + kPmBlock - 1) / kPmBlock); }

}  // namespace

hipError_t pm_deposit(const PmArgs &a, double *rho, hipStream_t st)
{
    if (a.n > 0)
        k_pm_deposit<<<(unsigned)((a.n + kPmChunk - 1) / kPmChunk), kPmBlock, 0, st>>>(a, grid_of(a), rho);
    return hipGetLastError();
}

hipError_t pm_green(int nside, float split_radius, float box, double2 *spec, hipStream_t st)
{
    // src/conv.f90:258-262: ismth2 = (2 pi smooth / box)^2, pref = box^2 / (pi N^3);
    // the mesh holds mass per cell, which the reference turns into a density
    // first: pmesh *= (NSIDEMESH / BOXSIZE)^3 in FP32 (src/partmesh.c:1797-1807),
    // folded into G here (the transform is linear)
    const double smooth = (double)split_radius, bx = (double)box;
    double ismth2 = 2.0 * kPiRef * smooth / bx;
    ismth2 = ismth2 * ismth2;
    const float rn1 = (float)nside / box;
    const float renormal = (rn1 * rn1) * rn1;
    const double pref = bx * bx / (kPiRef * (double)nside * (double)nside * (double)nside) * (double)renormal;
    const long long total = (long long)nside * nside * (nside / 2 + 1);
    k_pm_green<<<blocks_of(total), kPmBlock, 0, st>>>(nside, ismth2, pref, spec);
    return hipGetLastError();
}

hipError_t pm_interp(const PmArgs &a, const double *pot, double *grad, float *acc32, double *acc64,
                     hipStream_t st)
{
    const int N = a.nside;
    const double invx = (double)(float)(0.5 * (double)N / (double)a.box);   // src/partmesh.c:2596, FP32
    k_pm_gradient<<<dim3((unsigned)((N + kGradZ - 1) / kGradZ), (unsigned)((N + kGradY - 1) / kGradY), (unsigned)N),
                    dim3(kGradZ, kGradY), 0, st>>>(pot, N, invx, grad);
    if (a.n > 0)
        k_pm_interp<<<blocks_of(a.n), kPmBlock, 0, st>>>(a, grid_of(a), grad, acc32, acc64);
    return hipGetLastError();
}

hipError_t pm_zero(double *p, long long n, hipStream_t st)
{
    if (n > 0) {
        const long long b = (n + kPmBlock - 1) / kPmBlock;
        k_pm_zero<<<(unsigned)(b < 65536 ? b : 65536), kPmBlock, 0, st>>>(p, n);
    }
    return hipGetLastError();
}

}  // namespace pp2p
