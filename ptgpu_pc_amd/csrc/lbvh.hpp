// lbvh.hpp -- state of one LBVH build (the object behind the C ABI's ptgpu_clbvh handle).
#pragma once

#include <vector>

#include "common.hpp"

namespace ptgpu {
// Makes the handle's traversal layout current (tree height, four-wide nodes).  `recording`: the
// caller's stream is being recorded into a graph, so nothing may be read back.  `exact`: the caller
// needs the tree's height itself, not a bound checked on the device (exports, batch queries).  `wide` false:
// the four-wide nodes stay pending (the caller is about to change the tree).
int clbvh_prepare_traversal(ptgpu_clbvh *h, bool recording = false, bool exact = false, bool wide = true);
// Height bound of a traversal recorded before the height could be read back: the height last read
// for a build of the same kind (plain or optimised) plus this margin, or the default without one.
// An index-keyed tree's height is known without a read-back, so its frames wait for whether binary16 bounds blur it at the
// first build and at every 64th only (waiting at each costs a 97x61 frame with its rebuild 40 of 214 us); others take
// the last answer.  A handle set to skip the read-back waits for the first alone.
constexpr int kBlursAge = 64;
constexpr int kRecordedHeightMargin = 4;
constexpr int kRecordedHeightDefault = 41;   // the deepest tree the 64-entry four-wide stack walks
int clbvh_export_optimized(ptgpu_clbvh *h);

struct MItem;
// Scratch of the Morton-keyed traversal tree: each level's lists of leftover items, in two buffers by turns.
struct MortonScratch {
    int levels;
    int lists[8];      // lists of each level (kMMaxLevels)
    MItem *items[2];
    int *counts[2];
};
int clbvh_morton_scratch(ptgpu_clbvh *h, MortonScratch *m);
// Bound buffers handed between the level passes of the index-keyed refit (two halves of `per` floats).
int clbvh_level_scratch(ptgpu_clbvh *h, float **halves, size_t *per);
int clbvh_new(ptgpu_ctx *ctx, int n, ptgpu_clbvh **out);
// Handle state after a full build (bounds, Morton, topology, sort, refit) has been enqueued.
void clbvh_mark_built(ptgpu_clbvh *h);
}  // namespace ptgpu

struct ptgpu_clbvh {
    ptgpu_ctx *ctx = nullptr;
    int n = 0, cap = 0;
    int state = 0;            // 1 constructed (bounds+Morton), 2 radix tree, 3 BVH refit done
    int digit_bits = 8;       // radix-sort digit width (4 or 8)
    bool optimized = false;
    Shape *d_shapes = nullptr;
    ptgpu::DevBuf own_shapes;
    ptgpu::DevBuf boxes;                     // per-shape box records (input order) for the build's passes
    bool radix_pending = false;              // btn/btl topology not yet written (the refit writes it)
    ptgpu::DevBuf keysA, valsA, pairs;
    ptgpu::DevBuf btn, btl, tnodes, prims;
    ptgpu::DevBuf hist, status, misc;
    ptgpu::DevBuf lights, scan, opt_tmp;
    ptgpu::DevBuf mitems;                    // Morton-keyed traversal tree: leftover items of its levels
    ptgpu::DevBuf tnodes4;                   // four-wide view of tnodes, rebuilt after each refit
    bool wide_pending = false;
    ptgpu::DevBuf treelet;                   // treelet optimiser state (kept for the lazy export)
    bool export_pending = false;             // btn/btl still describe the tree before optimize
    int trav_topology = 1;    // traversal tree: 0 = the exported index-keyed tree, 1 = Morton-keyed LBVH
    bool height_pending = false;
    bool blurs_pending = false;   // acc.blurs is the previous build's
    int blurs_age = -1;           // builds since an answer was read (-1: none was)
    int known_height[2] = {0, 0};   // last heights read back: [0] plain build, [1] after optimize
    bool speculate = false;         // no read-back once a height is known: a bound, checked on the device
    unsigned *sorted = nullptr;
    int lights_for = -1, nlights = 0;
    ptgpu::DevAccel acc;
    std::vector<BVHNodeGPU> h_btn, h_btl;
    // misc: [0..5] scene centroid bounds, words 8.. counters ([0] unused, [1..8] sort
    // tile counters, [9] build error word, [10] binary16 bounds blur the tree, [11] traversal-tree height),
    // floats 64.. per-block bound partials
    float *scene6() const { return misc.as<float>(); }
    unsigned *counters() const { return misc.as<unsigned>() + 8; }
    float *partials() const { return misc.as<float>() + 64; }
    // device word holding the traversal tree's height (read back lazily by clbvh_prepare_traversal)
    unsigned *height_word() const { return counters() + 11; }
    // events: 0/1 morton, 2/3 topology, 4/5 sort, 5/6 refit, 7/8 optimize
    hipEvent_t ev[11] = {};   // 0-9 stage timing; 10: the traversal layout is ready (cross-stream use)
    bool timed[5] = {false, false, false, false, false};
};
