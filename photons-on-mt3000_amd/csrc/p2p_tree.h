// Host entry points of the device kd-tree build (internal to the library).
#pragma once
#include <hip/hip_runtime.h>

namespace pp2p {

constexpr int kSubMax = 4096;       // particles of a subtree built in one workgroup's LDS
constexpr int kSubLevels = 1024;    // levels of one subtree (the depth limit of a tree)
constexpr int kTreeTile = 4096;     // positions per block of the level passes
constexpr int kTreeUnitBytes = 64 * 24; // sums of a tile's samples, per group of 64
constexpr int kSubKid = 1 << 30;    // son codes from here on name subtrees

// Per-particle arrays of the build (n entries each, n + 1 where a caller
// reserves more).  The level passes and the subtrees share them: the
// subtrees' records go where the passes kept their lists, at the subtree's
// own particle range.
struct TreeScratch {
    int *x[3];      // coordinate planes, permuted in place
    int *idx;       // original index of the particle at each position
    int *la;        // level: misplaced particles of the left part; subtree: node id | (parent, side) << 12
    int *lb;        // level: misplaced particles of the right part; subtree: the two sons, 16 bits each
    int *lc;        // subtree: split value (float bits), by node
    int *ld;        // subtree: leaf ranges (start | length << 16)
};

// One level of the tree: segments of more than gmax particles.
struct TreeLevelView {
    int2 *seg;          // particle range (start, length)
    int *toff;          // first tile of each segment, the tile total last
    int2 *kid;          // sons: >= kSubKid subtree, >= 0 next-level segment, < 0 this level's leaf -(q + 1)
    int2 *leaf;         // this level's leaves (start, length)
    double *mean;
    float *split;
    int *left;          // particles of the left son
    int *swaps;         // misplaced pairs
    int2 *below;        // (nodes, leaves) below each segment
    int2 *idb;          // (node id, first leaf id) of each segment
    float4 *lo, *hi;    // box of each segment
};

// A subtree built by one workgroup.
struct TreeSub {
    int start, len, depth;
    int nnode, nleaf, nlev;     // nodes, leaves and levels of the subtree (nnode = -1: it did not fit)
    int id, leaf0;              // node id of its root, first leaf id
    float4 lo, hi;              // box of its root
};

// Device counters of the build.
struct TreeCounts {
    int nsub, misfit;           // subtrees; subtrees that did not fit
    int nseg[1025];             // segments of each level
};

// The finished tree: nodes by id, leaves by id.
struct TreeOut {
    int2 *son;
    float4 *node_center, *node_width;
    float4 *leaf_center, *leaf_width;
    int2 *leaf_rng;
    int *leaf_active;
};

// x planes and idx = 0..n-1 from n x 3 int32; the counters cleared and, when
// root is not null, level 0 set to the one segment [0, n), else sub 0 to it.
hipError_t tree_init(const int *posi, long long n, const TreeScratch &w, TreeCounts *counts, const TreeLevelView *root,
                     TreeSub *sub, hipStream_t st);
// One level (level < 1024): split values, partition (particles permuted in
// place), and the next level's segments, this level's leaves and the new
// subtrees.  cap: most segments the level can hold, tiles: most tiles.
// Per tile: csum one double, units kTreeUnitBytes, mask 64 words, tcnt and tmap one
// int.  More than subcap subtrees in all count as a misfit.
hipError_t tree_level(const TreeScratch &w, const TreeLevelView &lv, const TreeLevelView &nx, int level, int cap,
                      long long tiles, double int2pos, int maxleaf, int gmax, double *csum, void *units,
                      unsigned long long *mask, int *tcnt, int *tmap, TreeCounts *counts, TreeSub *sub, int subcap,
                      hipStream_t st);
// The subtrees: particles permuted in place, records and sizes; level
// offsets of subtree s at off[s * kSubLevels].
hipError_t tree_subs(const TreeScratch &w, TreeSub *sub, int nsub, double int2pos, int maxleaf, unsigned short *off,
                     TreeCounts *counts, hipStream_t st);
// The root's ids and box [lo, hi]: node 0 of level 0, or subtree 0 when root is null.
hipError_t tree_root(const TreeLevelView *root, TreeSub *sub, float4 lo, float4 hi, hipStream_t st);
hipError_t tree_below(const TreeLevelView &lv, int nseg, const int2 *below_next, const TreeSub *sub, hipStream_t st);
hipError_t tree_place(const TreeLevelView &lv, int nseg, const TreeLevelView &nx, int dir, TreeSub *sub,
                      const TreeOut &out, hipStream_t st);
hipError_t tree_place_subs(const TreeScratch &w, const TreeSub *sub, int nsub, const TreeOut &out, hipStream_t st);
// Target marking of the leaves and the FP64 positions in tree order.
hipError_t tree_finish(const TreeScratch &w, const TreeOut &out, int nleaf, const int *tag, double int2pos,
                       long long n, double *x3, hipStream_t st);

}  // namespace pp2p
