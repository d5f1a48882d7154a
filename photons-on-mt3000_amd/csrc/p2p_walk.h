// Host entry points of the device dual-tree walk (internal to the library).
#pragma once
#include <hip/hip_runtime.h>

namespace pp2p {

constexpr int kWalkTile = 256;      // fewest frames per tile of a round
constexpr int kWalkFrameBytes = 17; // of WalkFrames
constexpr int kWalkSmall = 1024;    // most tiles of that size; larger rounds have tiles of 1024 frames

// The kd-tree as the walk reads it.  son[k] = the two children of node k
// (>= 0: node id, < 0: leaf -(id + 1)); centres and widths of the node and
// leaf boxes (w unused); leaf_active >= 0 marks a leaf holding a local
// particle (a target).
struct WalkTree {
    const int2 *son;
    const float4 *node_center, *node_width;
    const float4 *leaf_center, *leaf_width;
    const int *leaf_active;
    int nnode, nleaf;
    float open_angle, cutoff;
};

// One cell in 32 bytes: node k at k, leaf l at nnode + l.
struct WalkCell {
    float cx, cy, cz;
    int a;                          // node: first son; leaf: active
    float wx, wy, wz;
    int b;                          // node: second son
};

// One round as the device keeps it: n opened frames at frame index fbase, its
// tiles at tbase; what their children are.
struct WalkRound {
    unsigned n;
    unsigned over;                  // 1: its frames did not fit the arrays (n is right)
    unsigned ticket;
    unsigned nsep;                  // well-separated children
    unsigned long long ntask;       // leaf-leaf children that are tasks
    long long fbase, tbase;
};

// The frames of all rounds, and per tile the look-back word and the
// exclusive count of well-separated children before it in its round.
struct WalkFrames {
    int2 *f;                        // (target, source) cells: >= 0 node, < 0 leaf -(id + 1)
    unsigned char *code;            // two bits per child: 0 none, 1 opened, 2 task, 3 well separated; bit 4 of a
                                    // frame with two children: the target cell was split
    unsigned *off;                  // first opened child in the next round
    int *cnt;                       // tasks at and below; then the first task's position
    long long cap;
    unsigned long long *look;
    int *sep;
    long long tcap;
};

hipError_t walk_cells(const WalkTree &t, WalkCell *cells, hipStream_t st);
// rounds[0] = cur (n frames at fbase, its tiles at tbase) with its counters
// cleared, rounds[1 .. count) cleared, and the tiles' look-back words from tbase
// on.  The frame of a first round (fbase 0) is set to the root's self pair.
hipError_t walk_begin(const WalkFrames &w, WalkRound *rounds, int count, const WalkRound &cur, hipStream_t st);
// Children of the round's frames: codes, offsets, the next round's frames and
// both rounds' counters, by up to `blocks` blocks.
hipError_t walk_open(const WalkTree &t, const WalkCell *cells, const WalkFrames &w, WalkRound *round, int blocks,
                     hipStream_t st);
// Backward: tasks at and below each of the n frames at fbase (children at fbase + n).
hipError_t walk_below(const WalkFrames &w, long long fbase, unsigned n, hipStream_t st);
// Positions: the first task of each opened child, the tasks of the round, and
// (nsep > 0) its well-separated pairs from ct / cs on, as cells (leaf id, or nleaf + node id).
hipError_t walk_emit(const WalkTree &t, const WalkCell *cells, const WalkFrames &w, long long fbase, long long tbase,
                     unsigned n, unsigned nsep, int *task_t, int *task_s, int *ct, int *cs, hipStream_t st);

}  // namespace pp2p
