// render.hip -- traversal engine and path-tracing megakernel for gfx950.
//
// Semantics follow rendering_kernel.cl (RadianceGPU :1072-1150, RadiancePathTracing :755-820,
// SampleLights :397-493, Intersect :194-363, IntersectP :375-395) in FP32 with every expression
// rounded as written (the library is built with -ffp-contract=off and IEEE division/sqrt).
//
// Differences from the reference that do not change results:
//   * Closest hit traverses a two-children-per-node layout (TNode) near-child first with the slab
//     test clipped to [0, t_best]; ties in t go to the higher shape index, which is exactly what
//     the brute-force loop (i = N-1 .. 0 with a strict <) returns.
//   * IntersectP is an any-hit traversal of the same tree that ignores shape N-1, the shape the
//     reference's brute-force loop never tests (Q10).
//   * SampleLights walks a precomputed list of the first lightCnt emitters in index order, drawing
//     the same random numbers in the same order as the reference's scan over all shapes.
//   * Persistent waves: each lane owns one pixel at a time and runs its spp samples back to back
//     (the running mean and RNG state stay in registers); a lane whose pixel is finished takes
//     the next pixel from a global counter, wave-wide through one atomic (ballot + popcount).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "lbvh.hpp"
#include "walk_half.hpp"

namespace ptgpu {

// One frame's work in a batch: a prepared tree, its scene and the frame's buffers (the reference's
// RadianceGPU arguments).
struct RenderJob {
    DevAccel acc;
    Vec *colors;
    unsigned *seeds;
    const Camera *camera;
    const Shape *shapes;
    const int *lights;
    int nlights;
    int width, height, currentSample, spp, max_depth;
    unsigned *pixels;
};

// A single-frame launch's shape (launch_shapes): workgroups that work, lanes of a wave that take pixels; the others help
// in the sparse phase.
struct LaunchShape {
    int blocks, lanes;
};
struct LaunchShapes {
    LaunchShape inside, outside;   // for a camera inside and outside the scene's box
};

struct RenderParams {
    DevAccel acc;
    Vec *colors;
    unsigned *seeds;
    const Camera *camera;
    const Shape *shapes;
    const int *lights;
    int nlights;
    const unsigned *lights_found; // single frames: device word with the emitters found; NULL: nlights is their number
    int width, height, currentSample, spp, max_depth;
    unsigned *pixels;
    unsigned long long *ray_counter;
    unsigned long long *trav_stats;
    unsigned *work_counter;
    int total;
    int regroup;
    int quad;                     // traversing lanes at or below which four lanes share each query
    const RenderJob *jobs;        // batch launches: job table, pixel prefix sums (njobs + 1)
    const unsigned *job_begin;
    int njobs;
    const int2 *tiles;            // tiled launches (RadianceBoxGPU): tile origins; NULL renders the whole frame
    int tile_w, tile_h;
    int slack;                    // half_slack of a tree whose height is known, for the classes that hold its walk.  (Computed in
                                  // the kernel it made KD frames 1 to 3% slower.)
    LaunchShapes launch;
    int depth_cap;                // deepest tree the launch's stack holds (checked when acc.height_check is set)
    const float *pack_tab;        // to_int_tab's table
    unsigned *status;             // the context's check words: [0] flags, [1] deepest height seen
};

// A launch recorded right after a build sized its stack for a height bound (acc.height_check set).
// The built tree is checked before any work: a build error (flag 1) or a tree deeper than the stack
// holds (flag 2) is recorded in the context's status words and the launch renders nothing.  Every
// thread reads the same words, so whole workgroups return together, before any barrier.
__device__ __forceinline__ bool recorded_tree_unfit(const RenderParams &P) {
    if (!P.acc.height_check) return false;
    const unsigned err = P.acc.height_check[0], h = P.acc.height_check[2];
    if (err == 0u && h <= (unsigned)P.depth_cap) return false;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicOr(P.status, err ? 1u : 2u);
        atomicMax(P.status + 1, h);
    }
    return true;
}

// The same check over a batch's jobs (P.status is set when some job's tree was recorded right after
// its build): the launch renders nothing if any job's tree does not fit.  Block-uniform: every block
// reads the same words and decides after one barrier.
__device__ bool recorded_jobs_unfit(const RenderParams &P) {
    __shared__ int s_unfit;
    if (threadIdx.x == 0) s_unfit = 0;
    __syncthreads();
    for (int j = threadIdx.x; j < P.njobs; j += blockDim.x) {
        const gmem<const unsigned> *hc = to_gmem(P.jobs[j].acc.height_check);
        if (!hc) continue;
        const unsigned err = hc[0], h = hc[2];
        if (err == 0u && h <= (unsigned)P.depth_cap) continue;
        atomicOr(&s_unfit, 1);
        if (blockIdx.x == 0) {
            atomicOr(P.status, err ? 1u : 2u);
            atomicMax(P.status + 1, h);
        }
    }
    __syncthreads();
    return s_unfit != 0;
}

// Whether the camera lies outside the scene's box (the union of the root node's child boxes).  Every thread
// reads the same words, so whole workgroups decide alike.
__device__ __forceinline__ bool camera_outside(const RenderParams &P) {
    const TNode4H &r = P.acc.nodes4h[P.acc.root];
    const float inf = __builtin_inff();
    f3 lo = mk(inf, inf, inf), hi = mk(-inf, -inf, -inf);
    for (int k = 0; k < 4; k++) {
        const uint4 c = r.c[k];   // an unused slot's inverted bounds change neither
        lo = mk(fminf(lo.x, half_lo(c.x)), fminf(lo.y, half_lo(c.y)), fminf(lo.z, half_lo(c.z)));
        hi = mk(fmaxf(hi.x, half_hi(c.x)), fmaxf(hi.y, half_hi(c.y)), fmaxf(hi.z, half_hi(c.z)));
    }
    const f3 o = ldvec(&P.camera->orig);
    return !(o.x >= lo.x && o.x <= hi.x && o.y >= lo.y && o.y <= hi.y && o.z >= lo.z && o.z <= hi.z);
}

// The frame pixel of claimed work item m: pixel m of the frame, or, in a tiled launch, pixel
// m % (tile_w * tile_h) of tile m / (tile_w * tile_h) in row-major order within the tile; -1 when a
// partial tile at the frame's right or bottom edge has no pixel there.
__device__ __forceinline__ int claimed_pixel(const RenderParams &P, unsigned m) {
    if (!P.tiles) return (int)m;
    const unsigned per = (unsigned)(P.tile_w * P.tile_h);
    const int2 o = P.tiles[m / per];
    const unsigned t = m % per;
    const int x = o.x + (int)(t % (unsigned)P.tile_w), y = o.y + (int)(t / (unsigned)P.tile_w);
    return (x < P.width && y < P.height) ? y * P.width + x : -1;
}

// The kernel's arguments, to be read where they are used: the shading pass of the per-lane-state kernel reads some
// forty words of them, which the compiler would load once and keep, and then has no scalar register left for
// the traversal loop (32 of them were spilled to lanes of a vector register, and 12 vector registers to scratch;
// so read, 7 and 8).  1024x768x16 of the 327,692-shape mesh 18.2 -> 17.75 ms, 640x480 of the 65,538-shape soup by
// RadianceGPU 2.25 -> 2.09, 97x61 of a 332-shape mesh 0.265 -> 0.250.
__device__ __forceinline__ cmem<RenderParams> *launch_args() {
    auto *p = (cmem<RenderParams> *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// the launch's lights
__device__ __forceinline__ int launch_lights(const RenderParams &P) {
    if (!P.lights_found) return P.nlights;
    const int found = __builtin_amdgcn_readfirstlane((int)*P.lights_found);
    return found < P.nlights ? found : P.nlights;
}

__device__ __forceinline__ void load_pack_table(const float *tab, float *s_pack) {
    for (int i = threadIdx.x; i < kPackEntries; i += blockDim.x) s_pack[i] = tab[i];
}
__global__ __launch_bounds__(256) void k_pack_table(float *tab) {
    const int k = threadIdx.x;
    unsigned lo = 0, hi = 0x3f800000u;   // least x (its bits) with to_int(x) >= k, by bisection
    while (lo < hi) {
        const unsigned mid = (lo + hi) >> 1;
        if (to_int(__uint_as_float(mid)) >= k) hi = mid; else lo = mid + 1;
    }
    tab[k] = k == 0 ? -__builtin_inff() : __uint_as_float(lo);
    if (k == 0) tab[256] = __builtin_inff();
}

// The path-tracing megakernel.  Lane state: one pixel (gid), its remaining samples, the RNG state
// and running mean; path state: ray, radiance, throughput, specularBounce, depth.
// BRUTE: no tree, and no more than kBrutePrims primitives: they, the first shapes and lights and the camera
// are read from LDS.
template <int STACK, bool STATS, bool BRUTE>
__global__ __launch_bounds__(256) void k_render(RenderParams P) {
    if (recorded_tree_unfit(P)) return;
    __shared__ int s_stack[BRUTE ? 1 : STACK * 256];
    __shared__ float s_pack[kPackEntries];
    load_pack_table(P.pack_tab, s_pack);
    int *stk = s_stack + threadIdx.x;
    const DevAccel &A = P.acc;
    const int nlights = launch_lights(P);
    constexpr int kLdsShapes = BRUTE ? 64 : 1, kLdsLights = BRUTE ? 32 : 1;
    __shared__ BruteScene<BRUTE ? kBrutePrims : 1> s_scene;
    __shared__ float s_shapes[kLdsShapes * 17], s_lights[kLdsLights * 14];
    __shared__ Camera s_cam;
    const Camera *cam = P.camera;
    if (BRUTE) {
        brute_stage(A.prims, A.nprims, s_scene);
        const int ns = A.nshapes < kLdsShapes ? A.nshapes : kLdsShapes;
        for (int i = threadIdx.x; i < ns * 17; i += blockDim.x)
            s_shapes[i] = reinterpret_cast<const float *>(P.shapes + i / 17)[i % 17];
        const int nl = nlights < kLdsLights ? nlights : kLdsLights;
        for (int i = threadIdx.x; i < nl * 14; i += blockDim.x) {
            const float *sw = reinterpret_cast<const float *>(P.shapes + P.lights[i / 14]);
            s_lights[i] = sw[i % 14 == 13 ? 25 : i % 14];
        }
        constexpr int kCamWords = (int)(sizeof(Camera) / sizeof(float));
        if ((int)threadIdx.x < kCamWords)
            reinterpret_cast<float *>(&s_cam)[threadIdx.x] = reinterpret_cast<const float *>(P.camera)[threadIdx.x];
        cam = &s_cam;
    }
    __syncthreads();
    unsigned long long spheres = 0;
    if (BRUTE) {
        const unsigned long long m = s_scene.spheres;
        spheres = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)m) |
                  ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(m >> 32)) << 32);
    }
    const unsigned long long lt = lanemask_lt();

    bool active = false, drained = false;
    int gid = 0, ci = 0, k = 0;
    unsigned s0 = 0, s1 = 0;
    f3 col = mk(0.f, 0.f, 0.f);
    f3 ro = mk(0.f, 0.f, 0.f), rd = mk(0.f, 0.f, 1.f), rad = mk(0.f, 0.f, 0.f), thr = mk(1.f, 1.f, 1.f);
    int spec = 1, depth = 0;
    unsigned long long n_closest = 0, n_any = 0;
    unsigned st_nodes = 0, st_prims = 0;
    unsigned *const pnv = STATS ? &st_nodes : nullptr;
    unsigned *const ppt = STATS ? &st_prims : nullptr;

    for (;;) {
        if (!drained) {
            const unsigned long long need = __ballot(!active);
            if (need) {
                const unsigned cnt = (unsigned)__popcll(need);
                const int leader = __ffsll((long long)need) - 1;
                unsigned base = 0;
                if ((int)__lane_id() == leader) base = atomicAdd(P.work_counter, cnt);
                base = __shfl(base, leader, kWave);
                if (base + cnt >= (unsigned)P.total) drained = true;
                if (!active) {
                    const unsigned my = base + (unsigned)__popcll(need & lt);
                    const int g = my < (unsigned)P.total ? claimed_pixel(P, my) : -1;
                    if (g >= 0) {   // (a tile pixel past the frame's edge: the lane claims again)
                        active = true;
                        gid = g;
                        const int x = gid % P.width, y = gid / P.width;
                        ci = (P.height - y - 1) * P.width + x;
                        s0 = P.seeds[2 * gid];
                        s1 = P.seeds[2 * gid + 1];
                        k = 0;
                        if (P.currentSample > 0) col = ldvec(P.colors + ci);
                        camera_ray(cam, s0, s1, P.width, P.height, x, y, ro, rd);
                        rad = mk(0.f, 0.f, 0.f); thr = mk(1.f, 1.f, 1.f); spec = 1; depth = 0;
                    }
                }
            }
        }
        if (__ballot(active) == 0) break;
        if (!active) continue;

        // ---- one path segment (RadianceOnePathTracing, rendering_kernel.cl:495-753) ----
        bool ended = false;
        if (depth > P.max_depth) {
            ended = true;
        } else {
            n_closest++;
            float t;
            const int id = BRUTE ? brute_closest_lds(s_scene, spheres, A.nprims, ro, rd, &t)
                                 : closest<STACK>(A, ro, rd, &t, stk, pnv, ppt);
            if (id < 0) {
                ended = true;
            } else {
                const f3 hp = add3(ro, smul(t, rd));
                Surface S;
                if (BRUTE && A.nshapes <= kLdsShapes) S = surface_of(s_shapes + id * 17, hp, rd);
                else S = surface_at(P.shapes + id, hp, rd);
                if (!iszero3(S.e)) {
                    if (spec) rad = add3(rad, mul3(thr, smul(fabsf(S.dp), S.e)));
                    ended = true;
                } else if (S.refl == DIFF) {
                    spec = 0;
                    thr = mul3(thr, S.c);
                    f3 Ld = mk(0.f, 0.f, 0.f);
                    for (int li = 0; li < nlights; li++) {
                        f3 sd, contrib;
                        float len;
                        bool shadow;
                        if (BRUTE && li < kLdsLights)
                            shadow = sample_light_words(s_lights + li * 14, s_lights[li * 14 + 13], s0, s1, hp, S.nl, &sd,
                                                        &len, &contrib);
                        else
                            shadow = sample_light(P.shapes + P.lights[li], s0, s1, hp, S.nl, &sd, &len, &contrib);
                        if (!shadow) continue;
                        n_any++;
                        const float maxt = len - kEpsilon;
                        const bool dark = BRUTE ? brute_any_lds(s_scene, spheres, A.nprims, hp, sd, maxt)
                                                : anyhit<STACK>(A, hp, sd, maxt, stk, pnv, ppt);
                        if (!dark) Ld = add3(Ld, contrib);
                    }
                    Ld = mul3(thr, Ld);
                    rad = add3(rad, Ld);
                    rd = diffuse_dir(S.nl, s0, s1);
                    ro = hp;
                } else {
                    spec = 1;
                    specular_or_refract(S, rd, thr, s0, s1);
                    ro = hp;
                }
                depth++;
            }
        }
        if (ended) {
            col = running_mean(col, rad, P.currentSample + k);
            k++;
            if (k < P.spp) {
                const int x = gid % P.width, y = gid / P.width;
                camera_ray(cam, s0, s1, P.width, P.height, x, y, ro, rd);
                rad = mk(0.f, 0.f, 0.f); thr = mk(1.f, 1.f, 1.f); spec = 1; depth = 0;
            } else {
                float *cp = reinterpret_cast<float *>(P.colors + ci);
                cp[0] = col.x; cp[1] = col.y; cp[2] = col.z;
                if (P.pixels) {
                    const int x = gid % P.width, y = gid / P.width;
                    P.pixels[y * P.width + x] = pack_rgba_tab(col, s_pack);
                }
                P.seeds[2 * gid] = s0;
                P.seeds[2 * gid + 1] = s1;
                active = false;
            }
        }
    }
    if (P.ray_counter) {
        // wave reduction, one atomic per wave
        unsigned long long a = n_closest, b = n_any;
        for (int o = 32; o > 0; o >>= 1) {
            a += __shfl_down(a, o, kWave);
            b += __shfl_down(b, o, kWave);
        }
        if (__lane_id() == 0) {
            atomicAdd(P.ray_counter, a);
            atomicAdd(P.ray_counter + 1, b);
        }
    }
    if (STATS && P.trav_stats) {
        unsigned long long a = st_nodes, b = st_prims;
        for (int o = 32; o > 0; o >>= 1) {
            a += __shfl_down(a, o, kWave);
            b += __shfl_down(b, o, kWave);
        }
        if (__lane_id() == 0) {
            atomicAdd(P.trav_stats, a);
            atomicAdd(P.trav_stats + 1, b);
        }
    }
}

// ---- megakernel with per-lane states ----
//
// The same paths as k_render, scheduled differently: every lane carries its own query (closest or
// any hit) and the wave advances all traversing lanes by one node per loop iteration.  A lane whose
// query ends does not hold the wave: it waits in a ready state until `regroup` lanes are ready (or
// none is traversing), then the wave runs one shading pass for exactly those lanes, each of which
// leaves it with its next query (or its pixel done).  The random numbers are drawn in the same
// order as in k_render (shadow-ray outcomes never draw), so the bits are the same.  Needs a tree
// whose root is an internal node (brute force and single-leaf trees run in k_render).
//
// What bounds it: on four workgroups per CU the instructions of the traversal step and of the shading
// pass (a timing copy counted 4,700 and 9,000 cycles a wave for them on a closed mesh, 45% and 33% of
// its time, before the pass was changed); on two, the latency of the longest pixels' steps (3,500 cycles
// beside one neighbour, 2,400 alone).  Hence:
//   * the step has no branch but the one around the triangle test: one fma per box plane (slab_hn) and the
//     children pushed by counted places (half_step); 265 -> 200 vector instructions;
//   * the traversal loop holds the step alone, so its back edge copies no path state;
//   * one shading pass serves a bounce: both lights and the next direction are drawn in it, and a finished
//     shadow ray starts the next query between passes;
//   * divisions and roots are correctly rounded in three and five instructions (rcp_exact, sqrt_exact);
//   * a wave with few queries left shares them among its lanes (half_sparse).
// Times before and after, one frame: 512x512x8 spp of the 65,538-shape soup 7.75 -> 5.1 ms; 1024x768x16 of the
// 327,692-shape mesh 36.0 -> 17.5 ms; 640x480x4 of a 20,492-shape SAH KD tree 5.0 -> 2.7 ms; 97x61x1 of a
// 332-shape mesh 0.57 -> 0.22 ms.
enum : int {
    kNeed = 0,    // wants a pixel
    kTrav = 1,    // traversing
    kADone = 2,   // any-hit query finished: bid >= 0 means occluded
    kCDone = 3,   // closest-hit query finished: tb / bid hold the result
    kLight = 4,   // next lights of SampleLights (from index li)
    kSeg = 5,     // start of a path segment (depth checked here)
    kEnded = 6,   // sample finished
    kIdle = 7,    // no work left
};
constexpr unsigned kShadowMin = 8;   // finished shadow rays that a full wave leaves the traversal loop for

template <int STACK, bool STATS, bool WIDE, bool MULTI, bool HALF, bool WAIT = false>
__global__ __launch_bounds__(256, HALF && !MULTI && STACK <= 36 ? 4 : HALF && STACK <= 48 ? 3 : 1) void k_render_lanes(RenderParams P) {
    if (!MULTI && recorded_tree_unfit(P)) return;
    if (MULTI && P.status && recorded_jobs_unfit(P)) return;
    LaunchShape shape = P.launch.inside;
    if (HALF && !MULTI &&
        (P.launch.outside.blocks != P.launch.inside.blocks || P.launch.outside.lanes != P.launch.inside.lanes) &&
        camera_outside(P))
        shape = P.launch.outside;
    if (!MULTI && (int)blockIdx.x >= shape.blocks) return;
    __shared__ int s_stack[STACK * 256];
    int *stk = s_stack + threadIdx.x;
    static_assert(!kIsShort<STACK> || (WIDE && HALF), "the short stack class serves the binary16 walk");
    const unsigned long long lt = lanemask_lt();
    // A single frame's first kLdsLights lights, 16 words each (words 0-12 of the light's Shape, then
    // its area), copied once per workgroup: SampleLights then reads LDS instead of two dependent
    // global loads (the light's index, then its Shape) per light in every shading pass.
    // The camera likewise: every new sample reads it.
    constexpr int kLdsLights = 32;
    __shared__ float s_lights[MULTI ? 16 : kLdsLights * 16];
    __shared__ Camera s_cam;
    __shared__ float s_pack[kPackEntries];
    load_pack_table(P.pack_tab, s_pack);
    int n_lds_lights = 0;
    const int p_nlights = MULTI ? 0 : launch_lights(P);
    if (!MULTI) {
        n_lds_lights = p_nlights < kLdsLights ? p_nlights : kLdsLights;
        for (int i = threadIdx.x; i < n_lds_lights * 16; i += blockDim.x) {
            const int l = i >> 4, w = i & 15;
            const float *sw = reinterpret_cast<const float *>(P.shapes + P.lights[l]);
            s_lights[i] = w <= 12 ? sw[w] : (w == 13 ? sw[25] : 0.f);
        }
        constexpr int kCamWords = (int)(sizeof(Camera) / sizeof(float));
        if ((int)threadIdx.x < kCamWords)
            reinterpret_cast<float *>(&s_cam)[threadIdx.x] = reinterpret_cast<const float *>(P.camera)[threadIdx.x];
        __syncthreads();
    }
    // A batch's first pixel per job (prefix sums of the jobs' pixel counts) for up to kLdsJobs jobs:
    // the search for a claimed pixel's job then reads LDS instead of one dependent global load per
    // halving.
    constexpr int kLdsJobs = 256;
    __shared__ unsigned s_job_begin[MULTI ? kLdsJobs : 1];
    if (MULTI) {
        const int nj = P.njobs < kLdsJobs ? P.njobs : kLdsJobs;
        for (int i = threadIdx.x; i < nj; i += blockDim.x) s_job_begin[i] = P.job_begin[i];
        __syncthreads();
    }
    // frame fields: the launch's own, or (batch) the lane's job's
    int jb = 0;
    // batch: the lane's job's fields that every shading pass reads, kept in registers from the pixel
    // claim on (a field read through the job table is one more dependent load)
    const gmem<const Shape> *j_shapes = to_gmem(P.shapes);
    const gmem<const int> *j_lights = to_gmem(P.lights);
    int j_nlights = p_nlights, j_max_depth = P.max_depth;
    // and those every new sample reads
    const gmem<const Camera> *j_camera = to_gmem(P.camera);
    int j_width = P.width, j_height = P.height, j_spp = P.spp, j_currentSample = P.currentSample;
    // the tree of the lane's current query (uniform for a single frame)
    const gmem<const TNode> *t_nodes = to_gmem(P.acc.nodes);
    const gmem<const TNode4> *t_nodes4 = to_gmem(P.acc.nodes4);
    HalfTree T;
    T.nodes = to_gmem(P.acc.nodes4h);
    T.prims = to_gmem(P.acc.prims);
    T.nprims = P.acc.nprims;
    T.skip = P.acc.nshapes - 1;
    int t_nnodes = P.acc.nnodes, t_root = P.acc.root;
    int t_slack = HALF && !MULTI ? P.slack : 0;   // (a batch's lanes take their job's)
    if (HALF && !MULTI && (kIsShort<STACK> || P.acc.height_check))
        t_slack = __builtin_amdgcn_readfirstlane(half_slack(STACK, P.acc));

    int st = (int)__lane_id() < shape.lanes ? kNeed : kIdle;
    bool drained = false;
    // Each wave's first pixels follow from its number; the counter deals out the rest, if there are any.  A frame that
    // is spread over 4,096 waves took 20 us of its 50 to 250 for their 8,192 turns at the counter.
    const unsigned first_deal = (blockIdx.x * 4 + threadIdx.x / kWave) * (unsigned)shape.lanes;
    const unsigned dealt = MULTI ? 0u : (unsigned)shape.blocks * 4u * (unsigned)shape.lanes;
    unsigned deal = __builtin_amdgcn_readfirstlane((int)(MULTI ? ~0u : first_deal));
    int gid = 0, k = 0, depth = 0, li = 0;
    bool spec = true;
    unsigned s0 = 0, s1 = 0;
    f3 col = mk(0.f, 0.f, 0.f), rad = col, thr = mk(1.f, 1.f, 1.f);
    f3 nl = col, Ld = col, contrib = col, inv = col;
    f3 rd2 = col, contrib2 = col;   // the bounce's second shadow ray, if `more`
    float maxt2 = 0.f;
    bool more = false;
    // the lane's query: HalfWalk's fields serve every node format (leaf and rs the binary16 one only)
    HalfWalk Q;
    Q.o = col;
    Q.d = mk(0.f, 0.f, 1.f);
    Q.tb = kInf;
    Q.bid = -1;
    Q.node = Q.sp = 0;
    Q.leaf = 0;
    Q.any = false;
    Q.rs = ray_slab(Q.o, mk(1.f, 1.f, 1.f));
    f3 &ro = Q.o, &rd = Q.d;
    float &tb = Q.tb;
    int &bid = Q.bid, &node = Q.node, &sp = Q.sp;
    bool &qany = Q.any;
    unsigned nv = 0;   // node visits (fp32 and binary nodes: a caller's tree may be malformed)
    unsigned long long n_closest = 0, n_any = 0;
    unsigned st_nodes = 0, st_prims = 0;

    // the primitives of one leaf for the lane's current query; true when an any-hit query is decided
    auto leaf = [&](int first, int cnt) -> bool {
        if (first < 0 || cnt > T.nprims - first) return false;   // malformed caller tree
        for (int q = 0; q < cnt; q++) {
            int id;
            const float t = prim_isect(from_gmem(T.prims), first + q, ro, rd, &id);
            if (STATS) st_prims++;
            if (qany) {
                if (t != 0.f && t < tb && id != T.skip) { bid = 1; return true; }
            } else if (t != 0.f && (t < tb || (t == tb && id > bid))) {
                tb = t;
                bid = id;
            }
        }
        return false;
    };
    // the lane's next query, along (ro, rd) as they stand at the end of the shading pass (tb = maxt for
    // any-hit): all lanes that leave the pass with one set it up together there
    bool fresh = false;
    auto start = [&](bool any, float maxt) {
        qany = any;
        tb = any ? maxt : kInf;
        st = kTrav;
        fresh = true;
    };
    auto set_up = [&]() {
        if (HALF) {
            half_start(Q, t_root);
        } else {
            bid = -1;
            inv = mk(1.0f / rd.x, 1.0f / rd.y, 1.0f / rd.z);
            node = t_root;
            sp = 0;
            nv = 0;
        }
        fresh = false;
    };

    // the light term joins the radiance and the path goes on along the direction drawn with it (nl holds it)
    auto end_bounce = [&]() {
        Ld = mul3(thr, Ld);
        rad = add3(rad, Ld);
        rd = nl;
        depth++;
        if (depth > (MULTI ? j_max_depth : P.max_depth)) {
            st = kEnded;
        } else {
            n_closest++;
            start(false, 0.f);
        }
    };

    // The wave's schedule.  The traversal loop changes the queries' state only and is left for everything
    // else, so that its back edge carries (and copies) nothing but that state.
    for (;;) {
        const unsigned long long live = __ballot(st != kIdle);
        if (!live) break;
        // a sparse wave (the end of the frame) shades sooner, so no lane's path waits long on others
        const unsigned nlive = (unsigned)__popcll(live);
        const unsigned quarter = (nlive + 3u) >> 2;
        unsigned regroup = (unsigned)P.regroup < quarter ? (unsigned)P.regroup : quarter;
        if (nlive >= 48u) regroup = (unsigned)P.regroup;
        const unsigned shadow_min = kShadowMin < regroup ? kShadowMin : regroup;
        const unsigned dense_min = HALF ? (unsigned)P.quad : 0u;
        // ---- traversal: one node of every traversing lane per iteration, until `regroup` lanes wait for
        // shading, `shadow_min` shadow rays have finished, or the wave is sparse ----
        for (;;) {
            const unsigned long long trav = __ballot(st == kTrav);
            if ((unsigned)__popcll(trav) <= dense_min || (unsigned)__popcll(live & ~trav) >= regroup ||
                (unsigned)__popcll(__ballot(st == kADone)) >= shadow_min)
                break;
            if (HALF && st == kTrav) {
                if (half_step<STACK, STATS, WAIT>(Q, T, stk, &st_nodes, &st_prims)) st = qany ? kADone : kCDone;
            }
            if (!WIDE && st == kTrav) {
                bool done = false;
                if ((unsigned)node >= (unsigned)t_nnodes || ++nv > kMaxVisits) {
                    done = true;   // malformed caller tree
                } else {
                    const TNode *np = from_gmem(t_nodes) + node;
                    const float4 a = np->a, b = np->b, c = np->c;
                    const int4 r = np->r;
                    if (STATS) st_nodes += 2;
                    float t0 = slab(a.x, a.y, a.z, a.w, b.x, b.y, ro, inv, tb);
                    float t1 = slab(b.z, b.w, c.x, c.y, c.z, c.w, ro, inv, tb);
                    if (r.x < 0 && t0 != __builtin_inff()) {
                        done = leaf(~r.x, r.z);
                        t0 = __builtin_inff();
                    }
                    if (!done && r.y < 0 && t1 != __builtin_inff()) {
                        done = leaf(~r.y, r.w);
                        t1 = __builtin_inff();
                    }
                    if (!done) {
                        const bool h0 = t0 != __builtin_inff(), h1 = t1 != __builtin_inff();
                        if (h0 && h1) {
                            const bool first0 = qany || t0 <= t1;
                            if (sp < STACK) stk[(sp++) * 256] = first0 ? r.y : r.x;
                            node = first0 ? r.x : r.y;
                        } else if (h0) {
                            node = r.x;
                        } else if (h1) {
                            node = r.y;
                        } else if (sp == 0) {
                            done = true;
                        } else {
                            node = stk[(--sp) * 256];
                        }
                    }
                }
                if (done) st = qany ? kADone : kCDone;
            }
            if (WIDE && !HALF && st == kTrav) {
                bool done = false;
                if ((unsigned)node >= (unsigned)t_nnodes || ++nv > kMaxVisits) {
                    done = true;   // malformed caller tree
                } else {
                    float4 lx, ly, lz, hx, hy, hz;
                    int4 rf, cn;
                    {
                        const TNode4 *np = from_gmem(t_nodes4) + node;
                        lx = np->lox; ly = np->loy; lz = np->loz;
                        hx = np->hix; hy = np->hiy; hz = np->hiz;
                        rf = np->ref;
                        cn = np->cnt;
                    }
                    constexpr float inf = __builtin_inff();
                    // branch-free: unused slots hold a box beyond every query's clip distance
                    float t0 = slab(lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, ro, inv, tb);
                    float t1 = slab(lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, ro, inv, tb);
                    float t2 = slab(lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, ro, inv, tb);
                    float t3 = slab(lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, ro, inv, tb);
                    if (STATS) st_nodes += (rf.x != kEmptyRef) + (rf.y != kEmptyRef) + (rf.z != kEmptyRef) +
                                           (rf.w != kEmptyRef);
                    // leaf children that are hit: their primitives now, one leaf per loop turn
                    unsigned lm = (rf.x < 0 && t0 != inf ? 1u : 0u) | (rf.y < 0 && t1 != inf ? 2u : 0u) |
                                  (rf.z < 0 && t2 != inf ? 4u : 0u) | (rf.w < 0 && t3 != inf ? 8u : 0u);
                    if (lm & 1u) t0 = inf;
                    if (lm & 2u) t1 = inf;
                    if (lm & 4u) t2 = inf;
                    if (lm & 8u) t3 = inf;
                    while (lm && !done) {
                        const unsigned k = (unsigned)__builtin_ctz(lm);
                        lm &= lm - 1u;
                        const int lr = k == 0 ? rf.x : k == 1 ? rf.y : k == 2 ? rf.z : rf.w;
                        const int lc = k == 0 ? cn.x : k == 1 ? cn.y : k == 2 ? cn.z : cn.w;
                        done = leaf(~lr, lc);
                    }
                    if (!done) {
                        // inner children: nearest first (order only changes the visit count)
                        int r0 = rf.x, r1 = rf.y, r2 = rf.z, r3 = rf.w;
                        auto cswap = [](float &ta, int &ra, float &tb_, int &rb) {
                            const bool sw = tb_ < ta;
                            const float tt = sw ? tb_ : ta;
                            tb_ = sw ? ta : tb_;
                            ta = tt;
                            const int rr = sw ? rb : ra;
                            rb = sw ? ra : rb;
                            ra = rr;
                        };
                        cswap(t0, r0, t1, r1);
                        cswap(t2, r2, t3, r3);
                        cswap(t0, r0, t2, r2);
                        cswap(t1, r1, t3, r3);
                        cswap(t1, r1, t2, r2);
                        if (t3 != inf && sp < STACK) stk[(sp++) * 256] = r3;
                        if (t2 != inf && sp < STACK) stk[(sp++) * 256] = r2;
                        if (t1 != inf && sp < STACK) stk[(sp++) * 256] = r1;
                        if (t0 != inf) node = r0;
                        else if (sp == 0) done = true;
                        else node = stk[(--sp) * 256];
                    }
                }
                if (done) st = qany ? kADone : kCDone;
            }
        }
        if (HALF) half_finish_overflowed<STACK, STATS>(Q, T, t_root, stk, &st_prims);
        // ---- finished shadow rays: the bounce's other shadow ray, or its next segment, both drawn when the
        // bounce was shaded, start here without a shading pass ----
        if (st == kADone) {
            if (bid < 0) Ld = add3(Ld, contrib);
            if (more) {
                more = false;
                contrib = contrib2;
                rd = rd2;
                n_any++;
                start(true, maxt2);
            } else if (li < j_nlights) {
                st = kLight;
            } else {
                end_bounce();
            }
            if (fresh) set_up();
        }
        {
            const unsigned long long trav = __ballot(st == kTrav);
            const unsigned ready = (unsigned)__popcll(live & ~trav);
            if (trav && ready < regroup) {
                // a sparse wave lends its idle lanes to the queries in flight
                if (HALF && (unsigned)__popcll(trav) <= (unsigned)P.quad &&
                    half_sparse<STACK, STATS, MULTI>(Q, T, t_slack, st == kTrav, trav, ready, regroup, s_stack,
                                                     &st_nodes, &st_prims))
                    st = qany ? kADone : kCDone;
                continue;
            }
        }
        cmem<RenderParams> *const args = launch_args();
        // ---- shading pass: pixels for lanes that need one (one atomic per wave) ----
        const unsigned long long need = __ballot(st == kNeed);
        if (need) {
            const unsigned cnt = (unsigned)__popcll(need);
            unsigned base = deal;
            if (deal != ~0u) {
                deal = ~0u;
                drained = dealt >= (unsigned)args->total;
            } else {
                const int leader = __ffsll((long long)need) - 1;
                if ((int)__lane_id() == leader) base = dealt + atomicAdd(args->work_counter, cnt);
                base = __shfl(base, leader, kWave);
                if (base + cnt >= (unsigned)args->total) drained = true;
            }
            if (st == kNeed) {
                const unsigned my = base + (unsigned)__popcll(need & lt);
                if (my < (unsigned)args->total) {
                    if (MULTI) {   // the job holding work item `my` (prefix sums of the jobs' pixel counts)
                        // two loops rather than one over a selected pointer, so the LDS search
                        // compiles to LDS reads (a pointer that may be either would be a flat one)
                        int lo = 0, hi = args->njobs - 1;
                        unsigned first;
                        if (args->njobs <= kLdsJobs) {
                            while (lo < hi) {
                                const int mid = (lo + hi + 1) >> 1;
                                if (s_job_begin[mid] <= my) lo = mid; else hi = mid - 1;
                            }
                            first = s_job_begin[lo];
                        } else {
                            const gmem<const unsigned> *jbg = to_gmem(args->job_begin);
                            while (lo < hi) {
                                const int mid = (lo + hi + 1) >> 1;
                                if (jbg[mid] <= my) lo = mid; else hi = mid - 1;
                            }
                            first = jbg[lo];
                        }
                        jb = lo;
                        gid = (int)(my - first);
                        // the job's tree, for every query of this pixel
                        const DevAccel &A = P.jobs[jb].acc;
                        t_nodes = to_gmem(A.nodes);
                        t_nodes4 = to_gmem(A.nodes4);
                        T.nodes = to_gmem(A.nodes4h);
                        T.prims = to_gmem(A.prims);
                        t_nnodes = A.nnodes;
                        T.nprims = A.nprims;
                        T.skip = A.nshapes - 1;
                        t_root = A.root;
                        t_slack = half_slack(STACK, A);
                        j_shapes = to_gmem(P.jobs[jb].shapes);
                        j_lights = to_gmem(P.jobs[jb].lights);
                        j_nlights = P.jobs[jb].nlights;
                        j_max_depth = P.jobs[jb].max_depth;
                        j_camera = to_gmem(P.jobs[jb].camera);
                        j_width = P.jobs[jb].width;
                        j_height = P.jobs[jb].height;
                        j_spp = P.jobs[jb].spp;
                        j_currentSample = P.jobs[jb].currentSample;
                    } else {
                        gid = claimed_pixel(P, my);
                    }
                    if (gid >= 0) {
                        const int W = (MULTI ? j_width : args->width), H = (MULTI ? j_height : args->height);
                        const int x = gid % W, y = gid / W;
                        s0 = to_gmem(MULTI ? P.jobs[jb].seeds : args->seeds)[2 * gid];
                        s1 = to_gmem(MULTI ? P.jobs[jb].seeds : args->seeds)[2 * gid + 1];
                        k = 0;
                        if ((MULTI ? j_currentSample : args->currentSample) > 0) {
                            const gmem<const float> *cv = reinterpret_cast<const gmem<const float> *>(
                                to_gmem(MULTI ? P.jobs[jb].colors : args->colors) + (H - y - 1) * W + x);
                            col = mk(cv[0], cv[1], cv[2]);
                        }
                        camera_ray(MULTI ? from_gmem(j_camera) : &s_cam, s0, s1, W, H, x, y, ro, rd);
                        rad = mk(0.f, 0.f, 0.f); thr = mk(1.f, 1.f, 1.f); spec = true; depth = 0;
                        st = kSeg;
                    } else {
                        st = drained ? kIdle : kNeed;   // a tile pixel past the frame's edge: claim again
                    }
                } else {
                    st = kIdle;
                }
            }
        }
        // ---- per-lane state machine until the lane holds a query or its pixel is done ----
        while (st >= kCDone && st <= kEnded) {
            if (st == kCDone) {
                if (bid < 0) {
                    st = kEnded;
                } else {
                    const f3 hp = add3(ro, smul(tb, rd));
                    const Surface S = surface_at((MULTI ? from_gmem(j_shapes) : args->shapes) + bid, hp, rd);
                    if (!iszero3(S.e)) {
                        if (spec) rad = add3(rad, mul3(thr, smul(fabsf(S.dp), S.e)));
                        st = kEnded;
                    } else if (S.refl == DIFF) {
                        spec = false;
                        thr = mul3(thr, S.c);
                        Ld = mk(0.f, 0.f, 0.f);
                        nl = S.nl;
                        ro = hp;
                        li = 0;
                        st = kLight;
                    } else {
                        spec = true;
                        specular_or_refract(S, rd, thr, s0, s1);
                        ro = hp;
                        depth++;
                        st = kSeg;
                    }
                }
            }
            if (st == kLight) {
                // The next two lights whose sample needs a shadow ray (the others only draw their random
                // numbers) and, once every light is drawn, the direction the path goes on in: shadow rays
                // never draw, so the numbers come in the reference's order, and one pass serves the whole
                // bounce.
                float len = 0.f;
                bool shoot = false;
                const int nlights = j_nlights;
                while (li < nlights && !more) {
                    f3 sd, con;
                    const bool sh = !MULTI && li < n_lds_lights
                                        ? sample_light_words(s_lights + 16 * li, s_lights[16 * li + 13], s0, s1, ro,
                                                             nl, &sd, &len, &con)
                                        : sample_light((MULTI ? from_gmem(j_shapes) : args->shapes) +
                                                           (MULTI ? from_gmem(j_lights) : args->lights)[li],
                                                       s0, s1, ro, nl, &sd, &len, &con);
                    li++;
                    if (!sh) continue;
                    if (shoot) {
                        more = true;
                        rd2 = sd;
                        contrib2 = con;
                        maxt2 = len - kEpsilon;
                    } else {
                        shoot = true;
                        rd = sd;
                        contrib = con;
                        tb = len - kEpsilon;
                    }
                }
                if (li >= nlights) nl = diffuse_dir(nl, s0, s1);
                if (shoot) {
                    n_any++;
                    start(true, tb);
                    continue;
                }
                end_bounce();
            }
            if (st == kSeg && depth > (MULTI ? j_max_depth : args->max_depth)) st = kEnded;
            if (st == kEnded) {
                col = running_mean(col, rad, (MULTI ? j_currentSample : args->currentSample) + k);
                k++;
                const int W = (MULTI ? j_width : args->width), H = (MULTI ? j_height : args->height);
                const int x = gid % W, y = gid / W;
                if (k < (MULTI ? j_spp : args->spp)) {
                    camera_ray(MULTI ? from_gmem(j_camera) : &s_cam, s0, s1, W, H, x, y, ro, rd);
                    rad = mk(0.f, 0.f, 0.f); thr = mk(1.f, 1.f, 1.f); spec = true; depth = 0;
                    st = kSeg;
                } else {
                    gmem<float> *cp = reinterpret_cast<gmem<float> *>(
                        to_gmem(MULTI ? P.jobs[jb].colors : args->colors) + (H - y - 1) * W + x);
                    cp[0] = col.x; cp[1] = col.y; cp[2] = col.z;
                    gmem<unsigned> *px = to_gmem(MULTI ? P.jobs[jb].pixels : args->pixels);
                    if (px) px[y * W + x] = pack_rgba_tab(col, s_pack);
                    gmem<unsigned> *sd = to_gmem(MULTI ? P.jobs[jb].seeds : args->seeds);
                    sd[2 * gid] = s0;
                    sd[2 * gid + 1] = s1;
                    st = drained ? kIdle : kNeed;
                }
            }
            if (st == kSeg) {
                n_closest++;
                start(false, 0.f);
            }
        }
        if (fresh) set_up();
    }
    cmem<RenderParams> *const args = launch_args();
    if (args->ray_counter) {
        unsigned long long a = n_closest, b = n_any;
        for (int o = 32; o > 0; o >>= 1) {
            a += __shfl_down(a, o, kWave);
            b += __shfl_down(b, o, kWave);
        }
        if (__lane_id() == 0) {
            atomicAdd(args->ray_counter, a);
            atomicAdd(args->ray_counter + 1, b);
        }
    }
    if (STATS && args->trav_stats) {
        unsigned long long a = st_nodes, b = st_prims;
        for (int o = 32; o > 0; o >>= 1) {
            a += __shfl_down(a, o, kWave);
            b += __shfl_down(b, o, kWave);
        }
        if (__lane_id() == 0) {
            atomicAdd(args->trav_stats, a);
            atomicAdd(args->trav_stats + 1, b);
        }
    }
}

// Batch queries (Intersect / IntersectP on arbitrary rays).
template <int STACK>
__global__ __launch_bounds__(256) void k_trace(DevAccel A, const Ray *rays, const float *maxt, int n, float *tout,
                                               int *idout, int *hitout, int any, unsigned *stats) {
    __shared__ int s_stack[STACK * 256];
    int *stk = s_stack + threadIdx.x;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float *rf = reinterpret_cast<const float *>(rays + i);
    const f3 o = mk(rf[0], rf[1], rf[2]), d = mk(rf[3], rf[4], rf[5]);
    unsigned nv = 0, pt = 0;
    if (any) {
        hitout[i] = anyhit<STACK>(A, o, d, maxt[i], stk, &nv, &pt) ? 1 : 0;
    } else {
        float t;
        const int id = closest<STACK>(A, o, d, &t, stk, &nv, &pt);
        tout[i] = id >= 0 ? t : 0.f;
        idout[i] = id;
    }
    if (stats) {
        atomicAdd(stats, nv);
        atomicAdd(stats + 1, pt);
    }
}

// The same queries over binary16 four-wide nodes.  A lane whose query ends takes the wave's next ray once eight
// lanes (or a quarter of those that still have work) have ended, so the wave's steps stay full, where one ray per
// thread over binary nodes let the longest of 64 hold the others; few rays are spread over all waves, whose idle
// lanes share them (half_sparse), and so is the end of a larger batch.  A wave's rays are fixed by its number, in
// runs of sixteen from all over the batch: neighbours in the batch often cost alike, and a counter that all waves
// take rays from cost more than it evened out (0.74 ms with one stretch a wave, 2 ms with the counter).  Bound by
// the step's instructions and its loads.  One million closest-hit and as many any-hit queries of a 65,538-shape
// soup, half of them from inside it in any direction: 1.42 -> 0.65 ms; 30,000: 0.53 -> 0.12; 1,000: 0.43 -> 0.063.
template <int STACK, bool WAIT>
__global__ __launch_bounds__(256, STACK <= 36 ? 4 : 2) void k_trace_half(DevAccel A, const Ray *rays, const float *maxt,
                                                                         int n, float *tout, int *idout, int *hitout,
                                                                         int any, int lanes, int regroup_max, int quad) {
    const int slack = __builtin_amdgcn_readfirstlane(half_slack(STACK, A));
    __shared__ int s_stack[STACK * 256];
    int *const stk = s_stack + threadIdx.x;
    HalfTree T;
    T.nodes = to_gmem(A.nodes4h);
    T.prims = to_gmem(A.prims);
    T.nprims = A.nprims;
    T.skip = A.nshapes - 1;
    const unsigned long long lt = lanemask_lt();
    // the wave's own share of the rays: every waves-th run of sixteen (of lanes, where fewer work)
    const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int run = lanes < 16 ? lanes : 16;
    const long long stride = (long long)gridDim.x * 4 * run;
    const int shift = __ffs(run) - 1;
    int next = 0;
    enum : int { kWant, kWalk, kDone, kOut };
    int st = (int)__lane_id() < lanes ? kWant : kOut;
    int cur = 0;
    HalfWalk W;
    W.o = W.d = mk(0.f, 0.f, 1.f);
    W.rs = ray_slab(W.o, W.d);
    W.tb = 0.f;
    W.bid = -1;
    W.node = W.leaf = W.sp = 0;
    W.any = any != 0;
    for (;;) {
        // results of the finished queries, then the next rays
        if (st == kDone) {
            half_finish_overflowed<STACK, false>(W, T, A.root, stk, nullptr);
            if (any) {
                hitout[cur] = W.bid >= 0 ? 1 : 0;
            } else {
                tout[cur] = W.bid >= 0 ? W.tb : 0.f;
                idout[cur] = W.bid;
            }
            st = kWant;
        }
        const unsigned long long want = __ballot(st == kWant);
        if (st == kWant) {
            const int p = next + (int)__popcll(want & lt);
            const long long at = (p >> shift) * stride + wave * run + (p & (run - 1));
            if (at < n) {
                cur = (int)at;
                const float *rf = reinterpret_cast<const float *>(rays + cur);
                W.o = mk(rf[0], rf[1], rf[2]);
                W.d = mk(rf[3], rf[4], rf[5]);
                W.tb = any ? maxt[cur] : kInf;
                half_start(W, A.root);
                st = kWalk;
            } else {
                st = kOut;
            }
        }
        next += (int)__popcll(want);
        const unsigned long long live = __ballot(st != kOut);
        if (!live) break;
        const unsigned quarter = ((unsigned)__popcll(live) + 3u) >> 2;
        const unsigned regroup = (unsigned)regroup_max < quarter ? (unsigned)regroup_max : quarter;
        unsigned long long walk;
        for (;;) {
            walk = __ballot(st == kWalk);
            if (__popcll(walk) <= quad || (unsigned)__popcll(live & ~walk) >= regroup) break;
            if (st == kWalk && half_step<STACK, false, WAIT>(W, T, stk, nullptr, nullptr)) st = kDone;
        }
        const unsigned ready = (unsigned)__popcll(live & ~walk);
        if (walk && ready < regroup &&
            half_sparse<STACK, false, false>(W, T, slack, st == kWalk, walk, ready, regroup, s_stack, nullptr, nullptr))
            st = kDone;
    }
}

// ---- scene preparation kernels ----
__global__ void k_index_prims(const Shape *shapes, int n, Prim *prims) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) prims[i] = prim_of(shapes + i, i, kLastInLeaf);
}

// A block's 4096 shapes, sixteen a thread, their emission loaded at once: bit q is shape base + 256 q + thread.
constexpr int kLightChunk = 4096;
__device__ __forceinline__ unsigned emitters(const Shape *shapes, int n, int base) {
    float e[16][3];
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int i = base + 256 * q + (int)threadIdx.x;
        const float *w = reinterpret_cast<const float *>(shapes + (i < n ? i : 0));
        e[q][0] = w[10]; e[q][1] = w[11]; e[q][2] = w[12];
    }
    asm volatile("" ::: "memory");   // compiler-only: the loads stay together
    unsigned m = 0;
#pragma unroll
    for (int q = 0; q < 16; q++)
        if (base + 256 * q + (int)threadIdx.x < n && !(e[q][0] == 0.f && e[q][1] == 0.f && e[q][2] == 0.f)) m |= 1u << q;
    return m;
}
__global__ __launch_bounds__(256) void k_light_count(const Shape *shapes, int n, unsigned *counts) {
    __shared__ unsigned s_c;
    if (threadIdx.x == 0) s_c = 0;
    __syncthreads();
    const unsigned c = (unsigned)__popc(emitters(shapes, n, blockIdx.x * kLightChunk));
    if (c) atomicAdd(&s_c, c);
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = s_c;
}
// The list itself and its length; a block starts after the emitters of the blocks before it (a single one needs no
// counts).  What bounds it for one frame's scene is its launch and two round trips: with the flags loaded one
// by one, a scan kernel between and the length read back, the nine shapes of a 256x256x4 frame took 42 of its then 192 us for the list.
__global__ __launch_bounds__(256) void k_light_write(const Shape *shapes, int n, const unsigned *counts, int cap,
                                                     int *out, unsigned *total) {
    __shared__ unsigned s_w[4][16], s_run;
    const int base = blockIdx.x * kLightChunk;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_run = 0;
    __syncthreads();
    unsigned before = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += 256) before += counts[b];
    if (before) atomicAdd(&s_run, before);
    const unsigned m = emitters(shapes, n, base);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const unsigned long long f = __ballot((m >> q) & 1u);
        if (lane == 0) s_w[w][q] = (unsigned)__popcll(f);
    }
    __syncthreads();
    unsigned run = s_run;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const unsigned long long f = __ballot((m >> q) & 1u);
        unsigned pos = run + (unsigned)__popcll(f & ((1ull << lane) - 1ull));
        for (int k = 0; k < 4; k++) {
            if (k < w) pos += s_w[k][q];
            run += s_w[k][q];
        }
        if (((m >> q) & 1u) && pos < (unsigned)cap) out[pos] = base + 256 * q + (int)threadIdx.x;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = run;
}

// TNode -> TNode4: the four grandchildren of binary node i (a leaf child is kept as it is).  Refs
// keep the binary numbering, so every internal node has a four-wide twin and a walk from the root
// that always takes two binary levels per step stays inside the array.  HALF: the binary16 copy (TNode4H)
// beside it (leaf counts dropped: leaves are runs ending in kLastInLeaf).
//
// One thread a node: three 64-byte loads, eight or twelve 16-byte stores, and the children's places by selects (an
// array filled by a running index went to scratch memory).  As two kernels, the second reading the first's nodes:
// 20.6 + 6.9 us for 65,537 nodes; as one: 9.7.
struct WideChild {
    float lx, ly, lz, hx, hy, hz;
    int ref, cnt;
};
template <bool HALF>
__device__ __forceinline__ void wide4_node(const TNode *__restrict__ bn, int nnodes, TNode4 *__restrict__ out,
                                           TNode4H *__restrict__ outh, int i) {
    if (i >= nnodes) return;
    auto left = [](const TNode &t) { return WideChild{t.a.x, t.a.y, t.a.z, t.a.w, t.b.x, t.b.y, t.r.x, t.r.z}; };
    auto right = [](const TNode &t) { return WideChild{t.b.z, t.b.w, t.c.x, t.c.y, t.c.z, t.c.w, t.r.y, t.r.w}; };
    const TNode t = bn[i];
    // (a ref outside the tree is kept, and the traversal rejects it)
    const bool il = t.r.x >= 0 && t.r.x < nnodes, ir = t.r.y >= 0 && t.r.y < nnodes;
    const TNode gl = bn[il ? t.r.x : i], gr = bn[ir ? t.r.y : i];
    // an unused slot is a point at 1e30: every query clips at t <= 1e20, so its slab test misses
    const WideChild none{kFarBox, kFarBox, kFarBox, kFarBox, kFarBox, kFarBox, kEmptyRef, 0};
    auto pick = [](bool first, const WideChild &x, const WideChild &y) {
        return WideChild{first ? x.lx : y.lx, first ? x.ly : y.ly, first ? x.lz : y.lz, first ? x.hx : y.hx,
                         first ? x.hy : y.hy, first ? x.hz : y.hz, first ? x.ref : y.ref, first ? x.cnt : y.cnt};
    };
    const WideChild r0 = pick(ir, left(gr), right(t)), r1 = pick(ir, right(gr), none);   // gr == t where !ir
    WideChild c[4];
    c[0] = pick(il, left(gl), left(t));
    c[1] = pick(il, right(gl), r0);
    c[2] = pick(il, r0, r1);
    c[3] = pick(il, r1, none);
    TNode4 o;
    o.lox = make_float4(c[0].lx, c[1].lx, c[2].lx, c[3].lx);
    o.loy = make_float4(c[0].ly, c[1].ly, c[2].ly, c[3].ly);
    o.loz = make_float4(c[0].lz, c[1].lz, c[2].lz, c[3].lz);
    o.hix = make_float4(c[0].hx, c[1].hx, c[2].hx, c[3].hx);
    o.hiy = make_float4(c[0].hy, c[1].hy, c[2].hy, c[3].hy);
    o.hiz = make_float4(c[0].hz, c[1].hz, c[2].hz, c[3].hz);
    o.ref = make_int4(c[0].ref, c[1].ref, c[2].ref, c[3].ref);
    o.cnt = make_int4(c[0].cnt, c[1].cnt, c[2].cnt, c[3].cnt);
    out[i] = o;
    if (HALF) {
        TNode4H h;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // a leaf without primitives has no run: stored as an unused slot
            const bool empty = c[k].ref == kEmptyRef || (c[k].ref < 0 && c[k].cnt <= 0);
            auto word = [&](float lo, float hi) {
                return empty ? kEmptyHalf : (unsigned)half_down(lo) | ((unsigned)half_up(hi) << 16);
            };
            h.c[k] = make_uint4(word(c[k].lx, c[k].hx), word(c[k].ly, c[k].hy), word(c[k].lz, c[k].hz),
                                empty ? ~0u : (unsigned)c[k].ref);
        }
        outh[i] = h;
    }
}
template <bool HALF>
__global__ __launch_bounds__(256) void k_wide4(const TNode *bn, int nnodes, TNode4 *out, TNode4H *outh) {
    wide4_node<HALF>(bn, nnodes, out, outh, blockIdx.x * blockDim.x + threadIdx.x);
}
// Several trees in one launch (a batch's after their build), described in the launch's arguments: 16 trees of 1,000 to
// 200,000 shapes, a launch each 128 us and their gaps, together 50 (the batch 5.31 -> 5.23 ms).
struct WideTable {
    static constexpr int kMax = 32;
    struct {
        const TNode *bn;
        TNode4 *out;
        int nnodes, first;   // first: the tree's first block
    } t[kMax];
    int n;
};
__global__ __launch_bounds__(256) void k_wide4_many(WideTable T) {
    int k = 0;
    while (k + 1 < T.n && (int)blockIdx.x >= T.t[k + 1].first) k++;
    wide4_node<true>(T.t[k].bn, T.t[k].nnodes, T.t[k].out, reinterpret_cast<TNode4H *>(T.t[k].out + T.t[k].nnodes),
                     ((int)blockIdx.x - T.t[k].first) * 256 + threadIdx.x);
}

// reference BVH layout -> TNode/Prim (child is a leaf iff nLeft == min / nRight == max)
__global__ void k_convert_bvh(const Shape *shapes, int n, const BVHNodeGPU *btn, const BVHNodeGPU *btl,
                              TNode *nodes, Prim *prims) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) prims[i] = prim_of(shapes + btl[i].nShape, btl[i].nShape, kLastInLeaf);   // one per leaf
    if (i < n - 1) {
        const int nl = btn[i].nLeft, nr = btn[i].nRight;
        const bool lleaf = nl == btn[i].min, rleaf = nr == btn[i].max;
        const Bound L = load_bound(lleaf ? &btl[nl].bound : &btn[nl].bound);
        const Bound R = load_bound(rleaf ? &btl[nr].bound : &btn[nr].bound);
        TNode t;
        t.a = make_float4(L.min_x, L.min_y, L.min_z, L.max_x);
        t.b = make_float4(L.max_y, L.max_z, R.min_x, R.min_y);
        t.c = make_float4(R.min_z, R.max_x, R.max_y, R.max_z);
        t.r = make_int4(lleaf ? ~nl : nl, rleaf ? ~nr : nr, lleaf ? 1 : 0, rleaf ? 1 : 0);
        nodes[i] = t;
    }
}

// Parents of a caller's reference-layout tree, taken from the child links the walk follows (the
// nParent fields are not trusted): par[i] for internal node i, par[n-1+k] for leaf k, -1 where no
// node points.  err[0] collects malformed links: 1 a child index out of range, 2 a node with two
// parents or a link back to the root.
__global__ void k_ref_parents(const BVHNodeGPU *btn, int n, int *par, unsigned *err) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int nl = btn[i].nLeft, nr = btn[i].nRight;
    const bool lleaf = nl == btn[i].min, rleaf = nr == btn[i].max;
    if ((unsigned)nl >= (unsigned)(lleaf ? n : n - 1) || (unsigned)nr >= (unsigned)(rleaf ? n : n - 1)) {
        atomicOr(err, 1u);
        return;
    }
    const int sl = lleaf ? n - 1 + nl : nl, sr = rleaf ? n - 1 + nr : nr;
    if (sl == 0 || sr == 0 || sl == sr) atomicOr(err, 2u);
    if (atomicExch(par + sl, i) != -1) atomicOr(err, 2u);
    if (sl != sr && atomicExch(par + sr, i) != -1) atomicOr(err, 2u);
}

// Height of that tree: the longest walk from a leaf up to the root (node 0), in edges, into err[1].
// A leaf no node points at sets err[0] bit 4; a walk longer than kMaxRefHeight (too deep for the
// traversal stack, or a cycle) sets bit 8; a leaf whose nShape is not a shape index sets bit 16.  err[2]: whether
// binary16 bounds blur the tree, from 64 leaves spread over it (half_blurs).
constexpr int kMaxRefHeight = 62;
__global__ __launch_bounds__(256) void k_ref_height(const BVHNodeGPU *btl, const int *par, int n, unsigned *err) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < kWave) {
        const Bound b = load_bound(&btl[(int)((long long)k * n / kWave)].bound);
        BlurSums s;
        s.add(b.min_x, b.min_y, b.min_z, b.max_x, b.max_y, b.max_z);
        const bool blurs = half_blurs(s);
        if (k == 0) err[2] = blurs ? 1u : 0u;
    }
    if (k >= n) return;
    if ((unsigned)btl[k].nShape >= (unsigned)n) atomicOr(err, 16u);
    int p = par[n - 1 + k], d = 1;
    while (p > 0 && d <= kMaxRefHeight) {
        p = par[p];
        d++;
    }
    if (p < 0) atomicOr(err, 4u);
    else if (p != 0) atomicOr(err, 8u);
    else atomicMax(err + 1, (unsigned)d);
}

// reference KD heap layout (1-based, children 2i/2i+1, leaves own kn[min..max)) -> TNode/Prim
__global__ void k_convert_kd(const Shape *shapes, const KDNodeGPU *kng, int kngCnt, const int *kn, int knCnt,
                             TNode *nodes, Prim *prims) {
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h < knCnt) prims[h] = prim_of(shapes + kn[h], kn[h], 0);   // caller ranges may overlap: no flags
    if (h >= 1 && h < kngCnt && kng[h].leaf == 0 && 2 * h + 1 < kngCnt) {
        const int cl = 2 * h, cr = 2 * h + 1;
        const bool lleaf = kng[cl].leaf == 1, rleaf = kng[cr].leaf == 1;
        const Bound L = load_bound(&kng[cl].bound), R = load_bound(&kng[cr].bound);
        TNode t;
        t.a = make_float4(L.min_x, L.min_y, L.min_z, L.max_x);
        t.b = make_float4(L.max_y, L.max_z, R.min_x, R.min_y);
        t.c = make_float4(R.min_z, R.max_x, R.max_y, R.max_z);
        t.r = make_int4(lleaf ? ~(int)kng[cl].min : cl, rleaf ? ~(int)kng[cr].min : cr,
                        lleaf ? (int)kng[cl].max - (int)kng[cl].min : 0,
                        rleaf ? (int)kng[cr].max - (int)kng[cr].min : 0);
        nodes[h] = t;
    }
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
int build_pack_table(ptgpu_ctx *ctx) {
    PT_TRY(ctx->pack_tab.ensure(kPackEntries * sizeof(float)));
    hipLaunchKernelGGL(k_pack_table, dim3(1), dim3(256), 0, ctx->stream, ctx->pack_tab.as<float>());
    PT_HIP(hipGetLastError());
    return PTGPU_OK;
}

int build_index_prims_into(ptgpu_ctx *ctx, const Shape *d_shapes, int n, Prim *prims) {
    hipLaunchKernelGGL(k_index_prims, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, d_shapes, n, prims);
    PT_HIP(hipGetLastError());
    return PTGPU_OK;
}

int build_index_prims(ptgpu_ctx *ctx, const Shape *d_shapes, int n, DevBuf &out_prims) {
    PT_TRY(out_prims.ensure((size_t)n * sizeof(Prim)));
    PT_TRY(build_index_prims_into(ctx, d_shapes, n, out_prims.as<Prim>()));
    return PTGPU_OK;
}

// one buffer: the fp32 four-wide nodes, then their binary16 copy
size_t wide_bytes(const DevAccel &acc) { return (size_t)(acc.nnodes > 0 ? acc.nnodes : 0) * (sizeof(TNode4) + sizeof(TNode4H)); }

int build_wide(ptgpu_ctx *ctx, DevAccel *acc, DevBuf &out_nodes4) {
    acc->nodes4 = nullptr;
    acc->nodes4h = nullptr;
    if (acc->mode == PTGPU_ACCEL_NONE || acc->root < 0 || acc->nnodes <= 0 || !acc->nodes) return PTGPU_OK;
    PT_TRY(out_nodes4.ensure(wide_bytes(*acc)));
    return build_wide_into(ctx, acc, out_nodes4.as<TNode4>());
}

int build_wide_into(ptgpu_ctx *ctx, DevAccel *acc, TNode4 *w4) {
    acc->nodes4 = nullptr;
    acc->nodes4h = nullptr;
    if (acc->mode == PTGPU_ACCEL_NONE || acc->root < 0 || acc->nnodes <= 0 || !acc->nodes) return PTGPU_OK;
    const size_t n4 = (size_t)acc->nnodes;
    const dim3 grid((unsigned)((n4 + 255) / 256));
    acc->nodes4 = w4;
    if (acc->leaf_runs) {
        acc->nodes4h = reinterpret_cast<TNode4H *>(w4 + n4);
        hipLaunchKernelGGL(k_wide4<true>, grid, dim3(256), 0, ctx->stream, acc->nodes, acc->nnodes, w4,
                           reinterpret_cast<TNode4H *>(w4 + n4));
    } else {
        hipLaunchKernelGGL(k_wide4<false>, grid, dim3(256), 0, ctx->stream, acc->nodes, acc->nnodes, w4, (TNode4H *)nullptr);
    }
    PT_HIP(hipGetLastError());
    return PTGPU_OK;
}

size_t light_scan_bytes(int n) { return ((size_t)((n + kLightChunk - 1) / kLightChunk) + 4) * 4; }

int build_light_list(ptgpu_ctx *ctx, const Shape *d_shapes, int n, int light_cnt, DevBuf &out, DevBuf &scan,
                     int *found, const unsigned **on_device) {
    *found = 0;
    if (on_device) *on_device = nullptr;
    if (light_cnt <= 0 || n <= 0) {
        PT_TRY(out.ensure(4));
        return PTGPU_OK;
    }
    PT_NO_CAPTURE(ctx, "building a light list");
    PT_TRY(scan.ensure(light_scan_bytes(n)));
    PT_TRY(out.ensure((size_t)light_cnt * 4));
    return build_light_list_into(ctx, d_shapes, n, light_cnt, out.as<int>(), scan.as<unsigned>(), found, on_device);
}

int build_light_list_into(ptgpu_ctx *ctx, const Shape *d_shapes, int n, int light_cnt, int *out, unsigned *scan,
                          int *found, const unsigned **on_device) {
    *found = 0;
    if (on_device) *on_device = nullptr;
    if (light_cnt <= 0 || n <= 0) return PTGPU_OK;
    PT_NO_CAPTURE(ctx, "building a light list");
    const int nb = (n + kLightChunk - 1) / kLightChunk;
    unsigned *counts = scan;
    unsigned *total = counts + nb;
    if (nb > 1) {
        hipLaunchKernelGGL(k_light_count, dim3(nb), dim3(256), 0, ctx->stream, d_shapes, n, counts);
        PT_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_light_write, dim3(nb), dim3(256), 0, ctx->stream, d_shapes, n, counts, light_cnt, out, total);
    PT_HIP(hipGetLastError());
    if (on_device) {
        *on_device = total;
        *found = light_cnt;
        return PTGPU_OK;
    }
    unsigned h_total = 0;
    PT_HIP(hipMemcpyAsync(&h_total, total, 4, hipMemcpyDeviceToHost, ctx->stream));
    PT_HIP(hipStreamSynchronize(ctx->stream));
    *found = (int)h_total < light_cnt ? (int)h_total : light_cnt;
    return PTGPU_OK;
}

size_t ref_parents_bytes(int n) { return (size_t)(n > 1 ? 2 * n - 1 : 1) * 4 + 64; }

int convert_bvh_ref(ptgpu_ctx *ctx, const Shape *d_shapes, int n, const BVHNodeGPU *d_btn, const BVHNodeGPU *d_btl,
                    DevBuf &nodes, DevBuf &prims, DevAccel *acc) {
    PT_TRY(ctx->tmp_parents.ensure(ref_parents_bytes(n)));
    PT_TRY(nodes.ensure((size_t)(n > 1 ? n - 1 : 1) * sizeof(TNode)));
    PT_TRY(prims.ensure((size_t)n * sizeof(Prim)));
    return convert_bvh_ref_into(ctx, d_shapes, n, d_btn, d_btl, nodes.as<TNode>(), prims.as<Prim>(),
                                ctx->tmp_parents.as<int>(), acc);
}

int convert_bvh_ref_into(ptgpu_ctx *ctx, const Shape *d_shapes, int n, const BVHNodeGPU *d_btn,
                         const BVHNodeGPU *d_btl, TNode *nodes, Prim *prims, int *parents, DevAccel *acc) {
    acc->depth = 0;
    if (n >= 2) {
        // The caller's links are checked before any kernel follows them, and the stack is sized from
        // the real height: a caller's tree (getTrees after optimize, or any other builder's) can be
        // much deeper than ceil(log2 n).
        PT_NO_CAPTURE(ctx, "measuring a caller's BVH");
        int *par = parents;
        unsigned *err = reinterpret_cast<unsigned *>(par + (2 * n - 1));
        PT_TRY(fill_u32(ctx->stream, par, 0xFFFFFFFFu, (size_t)(2 * n - 1)));
        PT_TRY(fill_u32(ctx->stream, err, 0u, 2));
        hipLaunchKernelGGL(k_ref_parents, dim3((n + 254) / 256), dim3(256), 0, ctx->stream, d_btn, n, par, err);
        PT_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_ref_height, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, d_btl, par, n, err);
        PT_HIP(hipGetLastError());
        unsigned h_err[3] = {0, 0, 0};
        PT_HIP(hipMemcpyAsync(h_err, err, 12, hipMemcpyDeviceToHost, ctx->stream));
        PT_HIP(hipStreamSynchronize(ctx->stream));
        PT_CHECK(!(h_err[0] & 3u), PTGPU_ERR_INVALID, "btn/btl: %s",
                 (h_err[0] & 1u) ? "a child index is out of range" : "a node has two parents (not a tree)");
        PT_CHECK(!(h_err[0] & 4u), PTGPU_ERR_INVALID, "btn/btl: a leaf is not reachable from the root");
        PT_CHECK(!(h_err[0] & 16u), PTGPU_ERR_INVALID, "btl: a leaf's nShape is out of range");
        PT_CHECK(!(h_err[0] & 8u), PTGPU_ERR_UNSUPPORTED, "btn/btl: tree deeper than %d levels (or cyclic)",
                 kMaxRefHeight);
        acc->depth = (int)h_err[1];
        acc->blurs = (int)h_err[2];
        acc->long_walks = 1;
    } else {
        PT_CHECK(n == 1, PTGPU_ERR_INVALID, "shapeCnt %d < 1", n);
        int ns = -1;
        PT_HIP(hipMemcpyAsync(&ns, &d_btl[0].nShape, 4, hipMemcpyDeviceToHost, ctx->stream));
        PT_HIP(hipStreamSynchronize(ctx->stream));
        PT_CHECK(ns == 0, PTGPU_ERR_INVALID, "btl: a leaf's nShape is out of range");
    }
    hipLaunchKernelGGL(k_convert_bvh, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, d_shapes, n, d_btn, d_btl,
                       nodes, prims);
    PT_HIP(hipGetLastError());
    acc->nodes = nodes;
    acc->prims = prims;
    acc->nprims = n;
    acc->nnodes = n - 1;
    acc->nshapes = n;
    acc->mode = PTGPU_ACCEL_BVH;
    acc->leaf_runs = 1;
    acc->root = n >= 2 ? 0 : ~0;
    acc->root_cnt = n >= 2 ? 0 : 1;
    return PTGPU_OK;
}

int convert_kd_ref(ptgpu_ctx *ctx, const Shape *d_shapes, int n, const KDNodeGPU *d_kng, int kngCnt, const int *d_kn,
                   int knCnt, DevBuf &nodes, DevBuf &prims, DevAccel *acc) {
    PT_CHECK(kngCnt >= 2, PTGPU_ERR_INVALID, "kngCnt %d < 2", kngCnt);
    PT_TRY(nodes.ensure((size_t)kngCnt * sizeof(TNode)));
    PT_TRY(prims.ensure((size_t)(knCnt > 0 ? knCnt : 1) * sizeof(Prim)));
    return convert_kd_ref_into(ctx, d_shapes, n, d_kng, kngCnt, d_kn, knCnt, nodes.as<TNode>(), prims.as<Prim>(), acc);
}

int convert_kd_ref_into(ptgpu_ctx *ctx, const Shape *d_shapes, int n, const KDNodeGPU *d_kng, int kngCnt,
                        const int *d_kn, int knCnt, TNode *nodes, Prim *prims, DevAccel *acc) {
    PT_CHECK(kngCnt >= 2, PTGPU_ERR_INVALID, "kngCnt %d < 2", kngCnt);
    PT_NO_CAPTURE(ctx, "converting a KD heap");
    const int m = kngCnt > knCnt ? kngCnt : knCnt;
    hipLaunchKernelGGL(k_convert_kd, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, d_shapes, d_kng, kngCnt, d_kn,
                       knCnt, nodes, prims);
    PT_HIP(hipGetLastError());
    KDNodeGPU root;
    PT_HIP(hipMemcpyAsync(&root, d_kng + 1, sizeof(KDNodeGPU), hipMemcpyDeviceToHost, ctx->stream));
    PT_HIP(hipStreamSynchronize(ctx->stream));
    acc->nodes = nodes;
    acc->prims = prims;
    acc->nprims = knCnt;
    acc->nnodes = kngCnt;
    acc->nshapes = n;
    acc->mode = PTGPU_ACCEL_KD;
    if (root.leaf == 1) {
        acc->root = ~(int)root.min;
        acc->root_cnt = (int)root.max - (int)root.min;
    } else {
        acc->root = 1;
        acc->root_cnt = 0;
    }
    int d = 0;
    while ((1ll << (d + 1)) < kngCnt) d++;
    acc->depth = d;
    return PTGPU_OK;
}

// four-wide walk: at most three pushes per visit and one visit per two binary levels; `least` raises
// the class for tests that run every stack instance on a shallow tree
static int stack_for_wide(const DevAccel &acc, int least) {
    int need = 3 * ((acc.depth + 2) / 2) + 1;
    if (need < least) need = least;
    if (need <= 32) return 32;
    if (need <= 48) return 48;   // 48 KB of LDS per workgroup: three workgroups per CU
    if (need <= 64) return 64;
    return -1;
}

// the deepest tree each stack holds (inverse of the two functions above and below)
static int wide_depth_cap(int stack) { return 2 * ((stack - 1) / 3) - 1; }
static int binary_depth_cap(int stack) { return stack - 2; }

static int stack_for(const DevAccel &acc, int least) {
    const int need = acc.mode == PTGPU_ACCEL_NONE ? 0 : acc.depth + 2;
    if (need <= 24 && least <= 24) return 24;
    if (need <= 64) return 64;
    return -1;
}

// Workgroups of a single-frame launch and the wave's share of pixels, for `total` work items.
//
// Set by the caller ("blocks_per_cu"): that many persistent workgroups per CU, never more than needed.
// By default, for the binary16 walk (the kernel looks where the camera is: it is device memory):
//   * In a small frame only the first 1, 2, 4 or 8 lanes of a wave take pixels and the others help their queries
//     (half_sparse): such a frame ends with its longest path whatever else runs, and shared queries take fewer
//     steps, each of which does more work.  (Times below in us: one frame alone, three in flight on a stream each.)
//     From outside much of a frame is background, so it is spread over all the waves that four workgroups per CU
//     hold, up to 8 pixels each (16 waves per CU: 32,768 pixels on 256 CUs): 180x180 of the 65,538-shape soup, 64
//     pixels a wave / eight: 831, 311 / 466, 213; at 256x256 eight halve the rate of a 20,482-shape mesh in flight.
//     Inside, every path is long.  Deep trees, KD trees and index-keyed or callers' trees, whose queries have many
//     steps or shapes to share, are spread alike; where walks are short (Morton-keyed trees of the 32-entry stack)
//     sharing saves one frame little and costs frames in flight much, so four pixels a wave end at 12,288 and eight
//     at 20,480.  64 pixels a wave / the share chosen: 6,592 pixels of a 332-shape mesh 399, 144 / 243, 141; 16,384 of a 5,132-shape
//     one 438, 170 / 413, 203, above the line 22,500 439, 174 (eight: 431, 265); 28,224 of a 20,492-shape one, deep,
//     490, 193 / 369, 255; 22,500 of the 5,132-shape one index-keyed 644, 259 / 496, 298, as a SAH KD tree
//     494, 188 / 356, 208, as a mean-split one 719, 269 / 379, 218.
//   * Larger frames get four workgroups per CU (what the registers and the stack leave room for), but a
//     frame of fewer than two pixels a lane (524,288 on 256 CUs) whose camera is outside the scene's box keeps
//     two.  Seen from inside, every pixel's path is long and more waves keep the SIMDs busy: 1024x768x16 of the
//     327,692-shape mesh, two / four a CU: 28.8 / 18.5 ms.  From outside, four are faster for a frame alone and
//     two for frames in flight, where another frame fills the drain and a build finds room, and the more so the
//     smaller the frame: the line lies where what the one loses is about what the other wins.  Two / four a CU,
//     8 spp, alone and three in flight (ms): 65,538-shape soup at 512x512 5.09 / 4.97 and 2.86 / 3.57, 720x720
//     6.93 / 6.51 and 4.15 / 5.50, above the line 800x800 8.04 / 6.78 and 4.91 / 6.16, 1024x1024 12.1 / 8.8 and
//     7.54 / 8.16; seen from further off, 512x512 7.36 / 6.00 and 4.43 / 5.38, 1024x768 16.4 / 11.4 and 10.4 / 11.1;
//     the 20,482-shape mesh from outside, 512x512 1.90 / 1.74 and 1.05 / 1.10, 720x720 2.93 / 2.59 and 1.69 / 1.79,
//     800x800 3.55 / 2.93 and 2.06 / 2.11; a 1,282-shape one at 512x512 1.49 / 1.29 and 0.82 / 0.81.  A caller who
//     keeps frames in flight sets two, at any size (900x600 of the soup: 3.2 against 4.8 ms).
static LaunchShapes launch_shapes(const ptgpu_ctx *ctx, const DevAccel &acc, int total, bool automatic, bool share) {
    const int cus = ctx->cu_count;
    const bool deep = stack_for_wide(acc, 0) != 32;
    auto shape = [&](int lanes, int per_cu) {
        const int all = cus * per_cu, need = (total + 4 * lanes - 1) / (4 * lanes);
        return LaunchShape{need < 1 ? 1 : need < all ? need : all, lanes};
    };
    if (!automatic) {
        const LaunchShape s = shape(kWave, ctx->blocks_per_cu);
        return LaunchShapes{s, s};
    }
    int in = kWave, out = kWave;
    if (share) {
        auto lanes = [&](int four, int eight) {
            return total <= 16 * cus ? 1 : total <= 32 * cus ? 2 : total <= four * cus ? 4 : total <= eight * cus ? 8 : kWave;
        };
        out = lanes(64, 128);
        in = acc.long_walks || deep ? out : lanes(48, 80);
    }
    return LaunchShapes{shape(in, 4), shape(out, out == kWave && total < 2 * 4 * 256 * cus ? 2 : 4)};
}

static bool walks_half(const ptgpu_ctx *ctx, const DevAccel &acc) {
    return (ctx->engine == 0 || ctx->engine == 3) && acc.mode != PTGPU_ACCEL_NONE && acc.root >= 0 && ctx->wide == 2 &&
           acc.nodes4h && !acc.blurs && stack_for_wide(acc, ctx->stack_min) > 0;
}

bool launch_spreads(const ptgpu_ctx *ctx, const DevAccel &acc, int pixels) {
    if (!walks_half(ctx, acc) || ctx->quad == 0) return false;
    const LaunchShapes s = launch_shapes(ctx, acc, pixels, true, true);
    return s.inside.lanes < kWave && s.outside.lanes < kWave;
}

int launch_render(ptgpu_ctx *ctx, const DevAccel &acc, const RenderLaunch &L) {
    // work items: every pixel, or every pixel slot of the listed tiles (slots past the frame's edge are skipped)
    const int total = L.tiles ? L.ntiles * L.tile_w * L.tile_h : L.width * L.height;
    if (total <= 0) return PTGPU_OK;
    const bool wf_ok = acc.mode != PTGPU_ACCEL_NONE && wf_supported(L.nlights) && !L.trav_stats && !L.tiles;
    if (ctx->engine == 2)
        PT_CHECK(wf_ok, PTGPU_ERR_UNSUPPORTED, "wavefront engine: needs a tree, <= 8 lights, no stats, no tiles");
    // the wavefront schedule only on request: one frame keeps at most W*H paths in flight, too few
    // to amortise its per-bounce barriers (measured 2x slower than the megakernels at 512x512)
    PT_CHECK(!(acc.height_check && ctx->engine == 2), PTGPU_ERR_UNSUPPORTED,
             "wavefront engine: a traversal recorded before the tree height was read back");
    if (wf_ok && ctx->engine == 2) return launch_render_wavefront(ctx, acc, L);
    const int st = stack_for(acc, ctx->stack_min);
    PT_CHECK(st > 0, PTGPU_ERR_UNSUPPORTED, "tree depth %d exceeds the 62-level traversal stack", acc.depth);
    unsigned *work_counter = L.work_counter;
    if (!work_counter) {
        PT_TRY(ctx->tmp_counter.ensure(64));
        work_counter = ctx->tmp_counter.as<unsigned>();
    }
    PT_TRY(fill_u32(ctx->stream, work_counter, 0u, 1));
    RenderParams P;
    P.acc = acc;
    P.colors = L.colors;
    P.seeds = L.seeds;
    P.camera = L.camera;
    P.shapes = L.shapes;
    P.lights = L.lights;
    P.nlights = L.nlights;
    P.lights_found = L.lights_found;
    P.width = L.width;
    P.height = L.height;
    P.currentSample = L.currentSample;
    P.spp = L.spp;
    P.max_depth = L.max_depth;
    P.pixels = L.pixels;
    P.ray_counter = L.ray_counter;
    P.trav_stats = L.trav_stats;
    P.work_counter = work_counter;
    P.pack_tab = ctx->pack_tab.as<float>();
    P.total = total;
    P.regroup = ctx->regroup;
    P.quad = ctx->quad;
    P.jobs = nullptr;
    P.job_begin = nullptr;
    P.njobs = 0;
    P.tiles = L.tiles;
    P.tile_w = L.tile_w;
    P.tile_h = L.tile_h;
    P.slack = 0;
    P.depth_cap = binary_depth_cap(st);
    P.status = nullptr;
    if (acc.height_check) {
        PT_TRY(ctx->rec_status.ensure(16));   // allocated at context creation; kept here for safety
        P.status = ctx->rec_status.as<unsigned>();
    }
    const bool lanes_engine = (ctx->engine == 0 || ctx->engine == 3) && acc.mode != PTGPU_ACCEL_NONE && acc.root >= 0;
    const bool half = walks_half(ctx, acc);
    // (counting launches keep one walk order for every shape)
    P.launch = launch_shapes(ctx, acc, total, ctx->blocks_auto && half, ctx->quad > 0 && !L.trav_stats);
    const int blocks = std::max(P.launch.inside.blocks, P.launch.outside.blocks);
    // auto and engine 3: per-lane states whenever there is a tree to walk (measured fastest at every
    // size tried); brute force and single-leaf scenes keep the lockstep megakernel
    if (lanes_engine) {
        int sw = acc.nodes4 && ctx->wide ? stack_for_wide(acc, ctx->stack_min) : -1;
        if (half && L.no_alloc && sw == 32) sw = 48;   // (the 32-entry class spills too, see below)
        if (sw > 0) P.depth_cap = wide_depth_cap(sw);
        // the binary16 walk of a tree in the 48-entry class runs on the short stack, four workgroups
        // per CU (short_stack 2, a test setting, runs every binary16 walk on the 8-entry class).  Held
        // to 128 registers, it and the 32-entry class keep seven or eight in scratch memory, which the
        // allocation-free entry does not ask the runtime for.
        const bool tiny = half && sw > 0 && ctx->short_stack == 2 && !L.no_alloc;
        const bool shortst = half && sw == 48 && ctx->short_stack == 1 && !L.no_alloc;
        P.slack = sw - 3 * ((acc.depth + 2) / 2);
#define PT_LANES(ST, STATS_, WIDE_, HALF_)                                                                      \
    hipLaunchKernelGGL((k_render_lanes<ST, STATS_, WIDE_, false, HALF_>), dim3(blocks), dim3(256), 0, ctx->stream, P)
#define PT_LANES_W(ST, STATS_) \
    do { if (half) PT_LANES(ST, STATS_, true, true); else PT_LANES(ST, STATS_, true, false); } while (0)
        if (tiny) {
            if (L.trav_stats) PT_LANES(kStackTiny, true, true, true);
            else PT_LANES(kStackTiny, false, true, true);
        } else if (half && acc.mode == PTGPU_ACCEL_KD && !L.trav_stats && (shortst || sw == 32)) {
            // leaves of several primitives (counting launches keep one walk order)
            if (shortst)
                hipLaunchKernelGGL((k_render_lanes<kStackShort, false, true, false, true, true>), dim3(blocks), dim3(256),
                                   0, ctx->stream, P);
            else
                hipLaunchKernelGGL((k_render_lanes<32, false, true, false, true, true>), dim3(blocks), dim3(256), 0,
                                   ctx->stream, P);
        } else if (shortst) {
            if (L.trav_stats) PT_LANES(kStackShort, true, true, true);
            else PT_LANES(kStackShort, false, true, true);
        } else if (sw > 0) {
            if (L.trav_stats) {
                if (sw == 32) PT_LANES_W(32, true);
                else if (sw == 48) PT_LANES_W(48, true);
                else PT_LANES_W(64, true);
            } else {
                if (sw == 32) PT_LANES_W(32, false);
                else if (sw == 48) PT_LANES_W(48, false);
                else PT_LANES_W(64, false);
            }
        } else if (L.trav_stats) {
            if (st == 24) PT_LANES(24, true, false, false);
            else PT_LANES(64, true, false, false);
        } else {
            if (st == 24) PT_LANES(24, false, false, false);
            else PT_LANES(64, false, false, false);
        }
#undef PT_LANES_W
#undef PT_LANES
    } else if (L.trav_stats) {
        if (st == 24) hipLaunchKernelGGL((k_render<24, true, false>), dim3(blocks), dim3(256), 0, ctx->stream, P);
        else hipLaunchKernelGGL((k_render<64, true, false>), dim3(blocks), dim3(256), 0, ctx->stream, P);
    } else if (acc.mode == PTGPU_ACCEL_NONE && acc.nprims <= kBrutePrims) {
        hipLaunchKernelGGL((k_render<24, false, true>), dim3(blocks), dim3(256), 0, ctx->stream, P);
    } else {
        if (st == 24) hipLaunchKernelGGL((k_render<24, false, false>), dim3(blocks), dim3(256), 0, ctx->stream, P);
        else hipLaunchKernelGGL((k_render<64, false, false>), dim3(blocks), dim3(256), 0, ctx->stream, P);
    }
    PT_HIP(hipGetLastError());
    return PTGPU_OK;
}

int launch_trace(ptgpu_ctx *ctx, const DevAccel &acc, unsigned int shapeCnt, const Ray *d_rays, const float *d_maxt,
                 int n, float *d_t, int *d_id, int *d_hit, bool any) {
    (void)shapeCnt;
    if (n <= 0) return PTGPU_OK;
    PT_CHECK(!acc.height_check, PTGPU_ERR_UNSUPPORTED,
             "batch queries cannot be recorded before the tree height was read back");
    const int sw = acc.nodes4h && !acc.blurs && acc.root >= 0 && ctx->wide == 2 ? stack_for_wide(acc, ctx->stack_min) : -1;
    if (sw > 0) {
        // Few rays are spread as launch_shapes spreads few pixels.  Four workgroups of the 32-entry stack on a CU
        // (five would fit: 0.80 against 0.71 ms for 20,000 shapes and a million rays); under the short stack, which
        // trees past 32 entries take, three for a batch that fills all lanes (0.64 against 0.72 ms for 65,538
        // shapes) and four for one that is spread (30,000 rays: 111 against 137 us).
        const int cus = ctx->cu_count;
        int lanes = 1;
        while (lanes < kWave && n > lanes * 16 * cus) lanes *= 2;
        if (lanes > 8 || ctx->quad == 0) lanes = kWave;
        const bool shortst = sw == 48 && ctx->short_stack != 0;
        const int per_cu = sw == 32 ? 4 : shortst ? (lanes == kWave ? 3 : 4) : sw == 48 ? 3 : 2;
        long long blocks = ((long long)n + 4 * lanes - 1) / (4 * lanes);
        if (blocks > (long long)cus * per_cu) blocks = (long long)cus * per_cu;
#define PT_TRACE_W(ST, WAIT)                                                                                          \
    hipLaunchKernelGGL((k_trace_half<ST, WAIT>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream, acc, d_rays, d_maxt, n, \
                       d_t, d_id, d_hit, any ? 1 : 0, lanes, 8, ctx->quad)
#define PT_TRACE(ST) \
    do { if (acc.mode == PTGPU_ACCEL_KD) PT_TRACE_W(ST, true); else PT_TRACE_W(ST, false); } while (0)
        if (sw == 32) PT_TRACE(32);
        else if (shortst) PT_TRACE(kStackShort);
        else if (sw == 48) PT_TRACE(48);
        else PT_TRACE(64);
#undef PT_TRACE
#undef PT_TRACE_W
        PT_HIP(hipGetLastError());
        return PTGPU_OK;
    }
    const int st = stack_for(acc, ctx->stack_min);
    PT_CHECK(st > 0, PTGPU_ERR_UNSUPPORTED, "tree depth %d exceeds the 62-level traversal stack", acc.depth);
    if (st == 24)
        hipLaunchKernelGGL(k_trace<24>, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, acc, d_rays, d_maxt, n, d_t,
                           d_id, d_hit, any ? 1 : 0, (unsigned *)nullptr);
    else
        hipLaunchKernelGGL(k_trace<64>, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, acc, d_rays, d_maxt, n, d_t,
                           d_id, d_hit, any ? 1 : 0, (unsigned *)nullptr);
    PT_HIP(hipGetLastError());
    return PTGPU_OK;
}

}  // namespace ptgpu

using namespace ptgpu;

// Resolve the traversal structure for (bvh, kd, shapes); NONE mode builds index-order prims.
static int resolve_accel(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const Shape *d_shapes, unsigned n,
                         DevAccel *acc, bool exact = false);

extern "C" int ptgpu_kdtree_device_accel(ptgpu_kdtree *kd, ptgpu::DevAccel *acc);

static int resolve_accel(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const Shape *d_shapes, unsigned n,
                         DevAccel *acc, bool exact) {
    PT_CHECK(!(bvh && kd), PTGPU_ERR_INVALID, "pass at most one of bvh / kd");
    if (bvh) {
        PT_CHECK(bvh->state >= 3, PTGPU_ERR_INVALID, "BVH not built (call build_bvh_tree)");
        PT_CHECK((unsigned)bvh->n == n, PTGPU_ERR_INVALID, "shapeCnt %u differs from the BVH's %d", n, bvh->n);
        PT_TRY(clbvh_prepare_traversal(bvh, ctx->capturing, exact));
        PT_CHECK(bvh->ctx->device == ctx->device, PTGPU_ERR_INVALID, "BVH built on device %d, render on device %d",
                 bvh->ctx->device, ctx->device);
        if (bvh->ctx != ctx && bvh->ctx->stream != ctx->stream) {
            // a handle built on another context's stream: this stream waits for that stream's work on
            // the handle (the build and the derived traversal layout) before it traverses
            PT_HIP(hipEventRecord(bvh->ev[10], bvh->ctx->stream));
            PT_HIP(hipStreamWaitEvent(ctx->stream, bvh->ev[10], 0));
        }
        *acc = bvh->acc;
        return PTGPU_OK;
    }
    if (kd) {
        PT_TRY(ptgpu_kdtree_device_accel(kd, acc));
        PT_CHECK((unsigned)acc->nshapes == n, PTGPU_ERR_INVALID, "shapeCnt %u differs from the KD tree's %d", n,
                 acc->nshapes);
        return PTGPU_OK;
    }
    PT_TRY(build_index_prims(ctx, d_shapes, (int)n, ctx->tmp_prims));
    acc->nodes = nullptr;
    acc->prims = ctx->tmp_prims.as<Prim>();
    acc->nprims = (int)n;
    acc->nnodes = 0;
    acc->nshapes = (int)n;
    acc->root = ~0;
    acc->root_cnt = (int)n;
    acc->depth = 0;
    acc->mode = PTGPU_ACCEL_NONE;
    return PTGPU_OK;
}

// RadianceGPU (box == NULL) and RadianceBoxGPU (box = {x, y, bwidth, bheight}) over reference-layout trees.
static int radiance_gpu_impl(ptgpu_ctx *ctx, int accel, const ptgpu_radiance_args *a, const int *box) {
    PT_CHECK(ctx && a, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(a->colors && a->seeds && a->camera && a->shapes && a->pixels, PTGPU_ERR_INVALID, "null buffer");
    PT_CHECK(a->shapeCnt >= 1, PTGPU_ERR_INVALID, "shapeCnt is 0");
    PT_CHECK(a->width > 0 && a->height > 0, PTGPU_ERR_INVALID, "bad frame size %dx%d", a->width, a->height);
    PT_CHECK((unsigned long long)a->width * (unsigned long long)a->height < (1ull << 30), PTGPU_ERR_UNSUPPORTED,
             "frame %dx%d: 2^30 pixels or more (seed indices 2*pixel must stay within int)", a->width,
             a->height);
    PT_CHECK(a->currentSample >= 0, PTGPU_ERR_INVALID, "currentSample < 0");
    PT_HIP(hipSetDevice(ctx->device));
    const int n = (int)a->shapeCnt;
    DevAccel acc;
    if (accel == PTGPU_ACCEL_BVH) {
        PT_CHECK(a->btn && a->btl, PTGPU_ERR_INVALID, "BVH mode needs btn and btl");
        PT_TRY(convert_bvh_ref(ctx, a->shapes, n, a->btn, a->btl, ctx->tmp_nodes, ctx->tmp_prims, &acc));
        PT_TRY(build_wide(ctx, &acc, ctx->tmp_nodes4));
    } else if (accel == PTGPU_ACCEL_KD) {
        PT_CHECK(a->kng && a->kn, PTGPU_ERR_INVALID, "KD mode needs kng and kn");
        PT_TRY(convert_kd_ref(ctx, a->shapes, n, a->kng, a->kngCnt, a->kn, a->knCnt, ctx->tmp_nodes, ctx->tmp_prims,
                              &acc));
        PT_TRY(build_wide(ctx, &acc, ctx->tmp_nodes4));
    } else {
        PT_CHECK(accel == PTGPU_ACCEL_NONE, PTGPU_ERR_INVALID, "unknown accel mode %d", accel);
        PT_TRY(resolve_accel(ctx, nullptr, nullptr, a->shapes, a->shapeCnt, &acc));
    }
    int nl = 0;
    RenderLaunch L;
    // (the wavefront engine sizes its queues by the number of lights)
    PT_TRY(build_light_list(ctx, a->shapes, n, (int)a->lightCnt, ctx->tmp_lights, ctx->tmp_scan, &nl,
                            ctx->engine == 2 ? nullptr : &L.lights_found));
    L.colors = a->colors;
    L.seeds = a->seeds;
    L.camera = a->camera;
    L.shapes = a->shapes;
    L.shapeCnt = a->shapeCnt;
    L.lights = ctx->tmp_lights.as<int>();
    L.nlights = nl;
    L.width = a->width;
    L.height = a->height;
    L.currentSample = a->currentSample;
    L.spp = 1;
    L.max_depth = ctx->max_depth;
    L.pixels = a->pixels;
    L.ray_counter = nullptr;
    L.trav_stats = nullptr;
    if (box) {   // the one box, as a one-entry tile list
        PT_TRY(ctx->tmp_tiles.ensure(64));
        PT_HIP(hipMemcpyAsync(ctx->tmp_tiles.p, box, 8, hipMemcpyHostToDevice, ctx->stream));
        L.tiles = ctx->tmp_tiles.as<int2>();
        L.ntiles = 1;
        L.tile_w = box[2];
        L.tile_h = box[3];
    }
    return launch_render(ctx, acc, L);
}

extern "C" {

int ptgpu_radiance_gpu(ptgpu_ctx *ctx, int accel, const ptgpu_radiance_args *a) {
    return radiance_gpu_impl(ctx, accel, a, nullptr);
}

int ptgpu_radiance_box_gpu(ptgpu_ctx *ctx, int accel, const ptgpu_radiance_args *a, int x, int y, int bwidth,
                           int bheight) {
    PT_CHECK(a, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(x >= 0 && y >= 0 && bwidth >= 1 && bheight >= 1 && x < a->width && y < a->height &&
                 (long long)bwidth * bheight < (1ll << 30),
             PTGPU_ERR_INVALID, "bad box (%d,%d) %dx%d in a %dx%d frame", x, y, bwidth, bheight, a->width, a->height);
    const int box[4] = {x, y, bwidth, bheight};
    return radiance_gpu_impl(ctx, accel, a, box);
}

}  // extern "C"

// ---------------------------------------------------------------------------------------------
// Allocation-free RadianceGPU (ptgpu_radiance_gpu_noalloc)
// ---------------------------------------------------------------------------------------------
namespace ptgpu {
constexpr size_t kNoAllocScratchBytes = size_t(128) << 20;
constexpr int kScratchDevices = 64;
}  // namespace ptgpu

// The work space of ptgpu_radiance_gpu_noalloc: the traversal layout converted from the caller's tree
// (binary nodes, primitives, four-wide nodes), the parent map of a caller's BVH, the light list and
// the persistent waves' pixel counter.  Each GPU holds its own copy until the process ends; host code
// reaches it only through the address hipGetSymbolAddress returns for that GPU.
static __device__ __align__(256) unsigned char scratch[ptgpu::kNoAllocScratchBytes];

namespace {
std::mutex g_scratch_mu;
void *g_scratch_ptr[ptgpu::kScratchDevices] = {};

// carves 256-byte-aligned pieces out of one device range
struct Carve {
    char *base;
    size_t used;
    template <class T> T *take(size_t bytes) {
        T *p = reinterpret_cast<T *>(base + used);
        used += (bytes + 255) & ~size_t(255);
        return p;
    }
};
size_t up256(size_t b) { return (b + 255) & ~size_t(255); }
}  // namespace

// Device address of this GPU's scratch array, looked up once per device with that device current
// (the context's set-up calls this; the entry point calls it again if the look-up failed then).
int ptgpu::noalloc_scratch_init(int device) {
    PT_CHECK(device >= 0 && device < kScratchDevices, PTGPU_ERR_UNSUPPORTED, "device %d: scratch table holds %d",
             device, kScratchDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return PTGPU_OK;
    void *ptr = nullptr;
    PT_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    PT_CHECK(ptr != nullptr, PTGPU_ERR_HIP, "hipGetSymbolAddress returned no address for the scratch array");
    g_scratch_ptr[device] = ptr;
    return PTGPU_OK;
}

extern "C" {

int ptgpu_radiance_gpu_noalloc(ptgpu_ctx *ctx, int accel, const ptgpu_radiance_args *a) {
    PT_CHECK(ctx && a, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(a->colors && a->seeds && a->camera && a->shapes && a->pixels, PTGPU_ERR_INVALID, "null buffer");
    PT_CHECK(a->shapeCnt >= 1 && a->shapeCnt < (1u << 30), PTGPU_ERR_INVALID, "shapeCnt %u out of range", a->shapeCnt);
    PT_CHECK(a->width > 0 && a->height > 0, PTGPU_ERR_INVALID, "bad frame size %dx%d", a->width, a->height);
    PT_CHECK((unsigned long long)a->width * (unsigned long long)a->height < (1ull << 30), PTGPU_ERR_UNSUPPORTED,
             "frame %dx%d: 2^30 pixels or more (seed indices 2*pixel must stay within int)", a->width, a->height);
    PT_CHECK(a->currentSample >= 0, PTGPU_ERR_INVALID, "currentSample < 0");
    PT_CHECK(accel == PTGPU_ACCEL_NONE || accel == PTGPU_ACCEL_BVH || accel == PTGPU_ACCEL_KD, PTGPU_ERR_INVALID,
             "unknown accel mode %d", accel);
    PT_CHECK(ctx->engine != 2, PTGPU_ERR_UNSUPPORTED,
             "the allocation-free entry runs the megakernel engines (the wavefront engine allocates its queues)");
    const int n = (int)a->shapeCnt;
    // the scratch this call needs, checked before any device work
    size_t nodes_b = 0, prims_b = 0, wide_b = 0, par_b = 0;
    if (accel == PTGPU_ACCEL_BVH) {
        PT_CHECK(a->btn && a->btl, PTGPU_ERR_INVALID, "BVH mode needs btn and btl");
        nodes_b = (size_t)(n > 1 ? n - 1 : 1) * sizeof(TNode);
        prims_b = (size_t)n * sizeof(Prim);
        wide_b = (size_t)(n > 1 ? n - 1 : 0) * (sizeof(TNode4) + sizeof(TNode4H));
        par_b = ref_parents_bytes(n);
    } else if (accel == PTGPU_ACCEL_KD) {
        PT_CHECK(a->kng && a->kn, PTGPU_ERR_INVALID, "KD mode needs kng and kn");
        PT_CHECK(a->kngCnt >= 2 && a->knCnt >= 0, PTGPU_ERR_INVALID, "kngCnt %d / knCnt %d", a->kngCnt, a->knCnt);
        nodes_b = (size_t)a->kngCnt * sizeof(TNode);
        prims_b = (size_t)(a->knCnt > 0 ? a->knCnt : 1) * sizeof(Prim);
        wide_b = (size_t)a->kngCnt * (sizeof(TNode4) + sizeof(TNode4H));
    } else {
        prims_b = (size_t)n * sizeof(Prim);
    }
    const size_t lights_b = (size_t)(a->lightCnt > 0 ? a->lightCnt : 1) * 4;
    const size_t need = up256(64) + up256(nodes_b) + up256(prims_b) + up256(wide_b) + up256(par_b) + up256(lights_b) +
                        up256(light_scan_bytes(n));
    PT_CHECK(need <= kNoAllocScratchBytes, PTGPU_ERR_UNSUPPORTED,
             "this frame's tree needs %zu bytes of scratch; the allocation-free entry holds %zu "
             "(ptgpu_radiance_gpu has no such limit)",
             need, kNoAllocScratchBytes);
    PT_HIP(hipSetDevice(ctx->device));
    PT_TRY(noalloc_scratch_init(ctx->device));
    Carve cv{static_cast<char *>(g_scratch_ptr[ctx->device]), 0};
    unsigned *counter = cv.take<unsigned>(64);
    TNode *nodes = cv.take<TNode>(nodes_b);
    Prim *prims = cv.take<Prim>(prims_b);
    TNode4 *wide = cv.take<TNode4>(wide_b);
    int *parents = cv.take<int>(par_b);
    int *lights = cv.take<int>(lights_b);
    unsigned *scan = cv.take<unsigned>(light_scan_bytes(n));
    DevAccel acc;
    if (accel == PTGPU_ACCEL_BVH) {
        PT_TRY(convert_bvh_ref_into(ctx, a->shapes, n, a->btn, a->btl, nodes, prims, parents, &acc));
        PT_TRY(build_wide_into(ctx, &acc, wide));
    } else if (accel == PTGPU_ACCEL_KD) {
        PT_TRY(convert_kd_ref_into(ctx, a->shapes, n, a->kng, a->kngCnt, a->kn, a->knCnt, nodes, prims, &acc));
        PT_TRY(build_wide_into(ctx, &acc, wide));
    } else {
        PT_TRY(build_index_prims_into(ctx, a->shapes, n, prims));
        acc.nodes = nullptr;
        acc.prims = prims;
        acc.nprims = n;
        acc.nnodes = 0;
        acc.nshapes = n;
        acc.root = ~0;
        acc.root_cnt = n;
        acc.depth = 0;
        acc.mode = PTGPU_ACCEL_NONE;
    }
    int nl = 0;
    PT_TRY(build_light_list_into(ctx, a->shapes, n, (int)a->lightCnt, lights, scan, &nl));
    RenderLaunch L;
    L.colors = a->colors;
    L.seeds = a->seeds;
    L.camera = a->camera;
    L.shapes = a->shapes;
    L.shapeCnt = a->shapeCnt;
    L.lights = lights;
    L.nlights = nl;
    L.width = a->width;
    L.height = a->height;
    L.currentSample = a->currentSample;
    L.spp = 1;
    L.max_depth = ctx->max_depth;
    L.pixels = a->pixels;
    L.ray_counter = nullptr;
    L.trav_stats = nullptr;
    L.work_counter = counter;
    L.no_alloc = true;
    return launch_render(ctx, acc, L);
}

}  // extern "C"

// Checks a ptgpu_render argument set, resolves its traversal structure and light list (the handle's
// prepared layout, or index-order primitives without a tree) and fills the launch description.
int ptgpu::prepare_render(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const ptgpu_render_args *a,
                          DevAccel *acc, RenderLaunch *L, bool lights_on_device) {
    PT_CHECK(ctx && a, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(a->colors && a->seeds && a->camera && a->shapes, PTGPU_ERR_INVALID, "null buffer");
    PT_CHECK(a->shapeCnt >= 1, PTGPU_ERR_INVALID, "shapeCnt is 0");
    PT_CHECK(a->width > 0 && a->height > 0, PTGPU_ERR_INVALID, "bad frame size %dx%d", a->width, a->height);
    PT_CHECK((unsigned long long)a->width * (unsigned long long)a->height < (1ull << 30), PTGPU_ERR_UNSUPPORTED,
             "frame %dx%d: 2^30 pixels or more (seed indices 2*pixel must stay within int)", a->width,
             a->height);
    PT_CHECK(a->spp >= 1 && a->currentSample >= 0, PTGPU_ERR_INVALID, "bad spp/currentSample");
    PT_CHECK(a->max_depth >= 0 && a->max_depth < 1024, PTGPU_ERR_INVALID, "bad max_depth");
    PT_HIP(hipSetDevice(ctx->device));
    PT_TRY(resolve_accel(ctx, bvh, kd, a->shapes, a->shapeCnt, acc));
    const int *lights = nullptr;
    int nl = 0;
    if (bvh) {
        if (bvh->lights_for != (int)a->lightCnt) {
            PT_TRY(build_light_list(ctx, a->shapes, (int)a->shapeCnt, (int)a->lightCnt, bvh->lights, bvh->scan,
                                    &bvh->nlights));
            bvh->lights_for = (int)a->lightCnt;
        }
        lights = bvh->lights.as<int>();
        nl = bvh->nlights;
    } else if (kd) {
        PT_TRY(kdtree_lights(kd, a->shapes, (int)a->shapeCnt, (int)a->lightCnt, &lights, &nl));
    } else {
        PT_TRY(build_light_list(ctx, a->shapes, (int)a->shapeCnt, (int)a->lightCnt, ctx->tmp_lights, ctx->tmp_scan,
                                &nl, lights_on_device && ctx->engine != 2 ? &L->lights_found : nullptr));
        lights = ctx->tmp_lights.as<int>();
    }
    L->colors = a->colors;
    L->seeds = a->seeds;
    L->camera = a->camera;
    L->shapes = a->shapes;
    L->shapeCnt = a->shapeCnt;
    L->lights = lights;
    L->nlights = nl;
    L->width = a->width;
    L->height = a->height;
    L->currentSample = a->currentSample;
    L->spp = a->spp;
    L->max_depth = a->max_depth;
    L->pixels = a->pixels;
    L->ray_counter = a->ray_counter;
    L->trav_stats = a->trav_stats;
    return PTGPU_OK;
}

int ptgpu::render_tiles(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const ptgpu_render_args *a,
                        const int2 *d_tiles, int ntiles, int tile_w, int tile_h, DevAccel *acc, RenderLaunch *L) {
    PT_CHECK(tile_w >= 1 && tile_h >= 1 && ntiles >= 0 && (long long)ntiles * tile_w * tile_h < (1ll << 30),
             PTGPU_ERR_INVALID, "bad tiles (%d of %dx%d)", ntiles, tile_w, tile_h);
    PT_TRY(prepare_render(ctx, bvh, kd, a, acc, L));
    if (ntiles == 0) return PTGPU_OK;
    PT_CHECK(d_tiles, PTGPU_ERR_INVALID, "null tile list");
    L->tiles = d_tiles;
    L->ntiles = ntiles;
    L->tile_w = tile_w;
    L->tile_h = tile_h;
    return launch_render(ctx, *acc, *L);
}

extern "C" {

int ptgpu_render(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const ptgpu_render_args *a) {
    DevAccel acc;
    RenderLaunch L;
    PT_TRY(prepare_render(ctx, bvh, kd, a, &acc, &L, true));
    return launch_render(ctx, acc, L);
}

int ptgpu_render_tiles(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const ptgpu_render_args *a,
                       const int *d_tile_origins, int ntiles, int tile_w, int tile_h) {
    DevAccel acc;
    RenderLaunch L;
    return render_tiles(ctx, bvh, kd, a, reinterpret_cast<const int2 *>(d_tile_origins), ntiles, tile_w, tile_h,
                        &acc, &L);
}

int ptgpu_render_batch(ptgpu_ctx *ctx, const ptgpu_render_job *jobs, int njobs, unsigned long long *d_ray_counter) {
    PT_CHECK(ctx && (jobs || njobs == 0) && njobs >= 0, PTGPU_ERR_INVALID, "null argument");
    if (njobs == 0) return PTGPU_OK;
    PT_HIP(hipSetDevice(ctx->device));
    ctx->batch.stream = ctx->stream;
    return launch_batch(ctx, ctx->batch, jobs, njobs, d_ray_counter);
}

}  // extern "C"

namespace ptgpu {
// The four-wide nodes of the jobs' LBVHs that were built on this context and not walked since (the others make theirs
// when they are resolved).
static int build_wide_many(ptgpu_ctx *ctx, const ptgpu_render_job *jobs, int njobs) {
    WideTable T;
    ptgpu_clbvh *hs[WideTable::kMax];
    int blocks = 0;
    T.n = 0;
    auto flush = [&]() -> int {
        if (T.n == 0) return PTGPU_OK;
        hipLaunchKernelGGL(k_wide4_many, dim3(blocks), dim3(256), 0, ctx->stream, T);
        PT_HIP(hipGetLastError());
        for (int k = 0; k < T.n; k++) {
            hs[k]->acc.nodes4 = T.t[k].out;
            hs[k]->acc.nodes4h = reinterpret_cast<TNode4H *>(T.t[k].out + T.t[k].nnodes);
            hs[k]->wide_pending = false;
        }
        T.n = 0;
        blocks = 0;
        return PTGPU_OK;
    };
    for (int j = 0; j < njobs; j++) {
        ptgpu_clbvh *h = jobs[j].bvh;
        if (!h || h->ctx != ctx || h->state < 3 || !h->wide_pending || h->height_pending) continue;
        if (h->acc.root < 0 || h->acc.nnodes <= 0 || !h->acc.nodes || !h->acc.leaf_runs) continue;
        bool listed = false;
        for (int k = 0; k < T.n; k++) listed = listed || hs[k] == h;
        if (listed) continue;
        PT_TRY(h->tnodes4.ensure(wide_bytes(h->acc)));
        hs[T.n] = h;
        T.t[T.n].bn = h->acc.nodes;
        T.t[T.n].out = h->tnodes4.as<TNode4>();
        T.t[T.n].nnodes = h->acc.nnodes;
        T.t[T.n].first = blocks;
        blocks += (h->acc.nnodes + 255) / 256;
        if (++T.n == WideTable::kMax) PT_TRY(flush());
    }
    return flush();
}

int launch_batch(ptgpu_ctx *ctx, BatchChannel &ch, const ptgpu_render_job *jobs, int njobs,
                 unsigned long long *d_ray_counter) {
    std::vector<RenderJob> table((size_t)njobs);
    std::vector<int> jst((size_t)njobs, 0);   // each job's traversal-stack class (32, 48 or 64 entries)
    if (!ctx->capturing) PT_TRY(build_wide_many(ctx, jobs, njobs));
    bool half = ctx->wide == 2;   // binary16 nodes only when every job's tree has them and none is blurred by them
    unsigned long long total = 0;
    for (int j = 0; j < njobs; j++) {
        const ptgpu_render_job &J = jobs[j];
        const ptgpu_render_args *a = &J.args;
        PT_CHECK(!!J.bvh != !!J.kd, PTGPU_ERR_INVALID, "job %d: pass exactly one of bvh / kd", j);
        for (int i = 0; i < j; i++)   // a handle holds one light list: jobs sharing it must agree on lightCnt
            PT_CHECK(!((jobs[i].bvh && jobs[i].bvh == J.bvh) || (jobs[i].kd && jobs[i].kd == J.kd)) ||
                         jobs[i].args.lightCnt == a->lightCnt,
                     PTGPU_ERR_INVALID, "jobs %d and %d share a tree but differ in lightCnt", i, j);
        PT_CHECK(a->colors && a->seeds && a->camera && a->shapes, PTGPU_ERR_INVALID, "job %d: null buffer", j);
        PT_CHECK(a->shapeCnt >= 2, PTGPU_ERR_UNSUPPORTED, "job %d: a batch needs at least two shapes per scene", j);
        PT_CHECK(a->width > 0 && a->height > 0, PTGPU_ERR_INVALID, "job %d: bad frame size %dx%d", j, a->width,
                 a->height);
        PT_CHECK((unsigned long long)a->width * (unsigned long long)a->height < (1ull << 30), PTGPU_ERR_UNSUPPORTED,
                 "job %d: frame %dx%d has 2^30 pixels or more", j, a->width, a->height);
        PT_CHECK(a->spp >= 1 && a->currentSample >= 0, PTGPU_ERR_INVALID, "job %d: bad spp/currentSample", j);
        PT_CHECK(a->max_depth >= 0 && a->max_depth < 1024, PTGPU_ERR_INVALID, "job %d: bad max_depth", j);
        RenderJob &R = table[(size_t)j];
        PT_TRY(resolve_accel(ctx, J.bvh, J.kd, a->shapes, a->shapeCnt, &R.acc));
        PT_CHECK(R.acc.root >= 0 && R.acc.nodes4, PTGPU_ERR_UNSUPPORTED, "job %d: the tree has no internal node", j);
        const int sw = stack_for_wide(R.acc, ctx->stack_min);
        PT_CHECK(sw > 0, PTGPU_ERR_UNSUPPORTED, "job %d: tree height %d exceeds the traversal stack", j, R.acc.depth);
        jst[(size_t)j] = sw;
        half = half && R.acc.nodes4h && !R.acc.blurs;
        if (J.bvh) {
            if (J.bvh->lights_for != (int)a->lightCnt) {
                PT_TRY(build_light_list(ctx, a->shapes, (int)a->shapeCnt, (int)a->lightCnt, J.bvh->lights,
                                        J.bvh->scan, &J.bvh->nlights));
                J.bvh->lights_for = (int)a->lightCnt;
            }
            R.lights = J.bvh->lights.as<int>();
            R.nlights = J.bvh->nlights;
        } else {
            PT_TRY(kdtree_lights(J.kd, a->shapes, (int)a->shapeCnt, (int)a->lightCnt, &R.lights, &R.nlights));
        }
        R.colors = a->colors;
        R.seeds = a->seeds;
        R.camera = a->camera;
        R.shapes = a->shapes;
        R.width = a->width;
        R.height = a->height;
        R.currentSample = a->currentSample;
        R.spp = a->spp;
        R.max_depth = a->max_depth;
        R.pixels = a->pixels;
        total += (unsigned long long)a->width * (unsigned long long)a->height;
        PT_CHECK(total < (1ull << 31), PTGPU_ERR_UNSUPPORTED, "batch of more than 2^31 pixels");
    }
    // At most two launches, run at once on the channel's stream and one forked from it.  The kernel's
    // registers allow three workgroups per CU and so does a 48-entry stack (50 KB), so every tree but the
    // deepest shares one launch sized for the deepest of them; trees that need 64 entries (two workgroups per
    // CU) get a launch of their own rather than hold the whole batch at that.  The launches share the CUs'
    // workgroups by their samples: each asking for all of them ran one launch's workgroups only when the
    // other's had ended (16 scenes in two launches of three per CU each 7.6 ms, in one 5.2).
    struct Cls {
        int st;
        std::vector<int> jobs;
        unsigned long long total, samples;
        bool checks;
        size_t jo, bo;   // offsets of its jobs and its prefix sums in the table image
    };
    std::vector<Cls> cls;
    unsigned long long samples = 0;
    for (int c : {64, 48}) {
        Cls K{c == 64 ? 64 : 32, {}, 0, 0, false, 0, 0};
        for (int j = 0; j < njobs; j++)
            if ((jst[(size_t)j] == 64) == (c == 64)) {
                const RenderJob &R = table[(size_t)j];
                const unsigned long long px = (unsigned long long)R.width * (unsigned long long)R.height;
                if (jst[(size_t)j] > K.st) K.st = jst[(size_t)j];
                K.jobs.push_back(j);
                K.total += px;
                K.samples += px * (unsigned long long)R.spp;
                K.checks = K.checks || R.acc.height_check;
            }
        // Lanes take pixels in this order: the longest chains (most samples) first, so the launch does not end
        // waiting on one started late; then the smaller frames, so that it ends in the many bottom rows of a
        // large one, which are often background (16 scenes, small / large frames last: 6.9 / 5.7 ms).
        std::stable_sort(K.jobs.begin(), K.jobs.end(), [&](int x, int y) {
            const RenderJob &X = table[(size_t)x], &Y = table[(size_t)y];
            if (X.spp != Y.spp) return X.spp > Y.spp;
            return (long long)X.width * X.height < (long long)Y.width * Y.height;
        });
        samples += K.samples;
        if (!K.jobs.empty()) cls.push_back(std::move(K));
    }
    size_t img_bytes = 0;
    for (Cls &K : cls) {
        K.jo = img_bytes;
        img_bytes = (K.jo + K.jobs.size() * sizeof(RenderJob) + 63) & ~size_t(63);
        K.bo = img_bytes;
        img_bytes = (K.bo + (K.jobs.size() + 1) * sizeof(unsigned) + 63) & ~size_t(63);
    }
    std::vector<char> img(img_bytes, 0);
    for (Cls &K : cls) {
        unsigned run = 0;
        for (size_t q = 0; q < K.jobs.size(); q++) {
            const RenderJob &R = table[(size_t)K.jobs[q]];
            std::memcpy(img.data() + K.jo + q * sizeof(RenderJob), &R, sizeof(RenderJob));
            std::memcpy(img.data() + K.bo + q * sizeof(unsigned), &run, sizeof(unsigned));
            run += (unsigned)(R.width * R.height);
        }
        std::memcpy(img.data() + K.bo + K.jobs.size() * sizeof(unsigned), &run, sizeof(unsigned));
    }
    hipStream_t stream = ch.stream;
    if (!ch.copied) PT_HIP(hipEventCreateWithFlags(&ch.copied, hipEventDisableTiming));
    if (!ch.ready) PT_HIP(hipEventCreateWithFlags(&ch.ready, hipEventDisableTiming));
    if (stream != ctx->stream) {   // builds and layout conversion ran on the context's stream
        PT_HIP(hipEventRecord(ch.ready, ctx->stream));
        PT_HIP(hipStreamWaitEvent(stream, ch.ready, 0));
    }
    void *d_table = nullptr;
    if (ctx->capturing) {
        // recorded: the table gets a pinned copy and a device buffer of its own, kept with the graph
        PT_TRY(record_stage(ctx, stream, img.data(), img_bytes, img_bytes, &d_table));
    } else {
        // stage the table through pinned memory; the channel's previous copy must be done before reuse
        PT_HIP(hipEventSynchronize(ch.copied));
        if (ch.pinned_bytes < img_bytes) {
            if (ch.pinned) PT_HIP(hipHostFree(ch.pinned));
            ch.pinned = nullptr;
            ch.pinned_bytes = 0;
            PT_HIP(hipHostMalloc(&ch.pinned, img_bytes * 2, hipHostMallocDefault));
            ch.pinned_bytes = img_bytes * 2;
        }
        std::memcpy(ch.pinned, img.data(), img_bytes);
        PT_TRY(ch.table.ensure(img_bytes));
        PT_HIP(hipMemcpyAsync(ch.table.p, ch.pinned, img_bytes, hipMemcpyHostToDevice, stream));
        PT_HIP(hipEventRecord(ch.copied, stream));
        d_table = ch.table.p;
    }
    const int ncls = (int)cls.size();
    PT_TRY(ch.counter.ensure((size_t)64 * ncls));
    PT_TRY(fill_u32(stream, ch.counter.p, 0u, (size_t)16 * ncls));   // one work counter per class, 64 B apart
    if (ncls > 1) {
        if (!ch.fork) PT_HIP(hipEventCreateWithFlags(&ch.fork, hipEventDisableTiming));
        PT_HIP(hipEventRecord(ch.fork, stream));
    }
    for (int k = 0; k < ncls; k++) {
        const Cls &K = cls[(size_t)k];
        hipStream_t s = stream;
        if (k > 0) {
            if (!ch.sub) PT_HIP(hipStreamCreateWithFlags(&ch.sub, hipStreamNonBlocking));
            if (!ch.join) PT_HIP(hipEventCreateWithFlags(&ch.join, hipEventDisableTiming));
            s = ch.sub;
            PT_HIP(hipStreamWaitEvent(s, ch.fork, 0));
        }
        RenderParams P;
        std::memset(static_cast<void *>(&P), 0, sizeof(P));
        P.acc = table[(size_t)K.jobs[0]].acc;   // unused by the batch variant
        P.ray_counter = d_ray_counter;
        P.trav_stats = nullptr;
        P.work_counter = ch.counter.as<unsigned>() + 16 * k;
        P.pack_tab = ctx->pack_tab.as<float>();
        P.total = (int)K.total;
        P.regroup = ctx->batch_regroup;
        P.quad = ctx->quad;
        P.jobs = reinterpret_cast<const RenderJob *>(static_cast<char *>(d_table) + K.jo);
        P.job_begin = reinterpret_cast<const unsigned *>(static_cast<char *>(d_table) + K.bo);
        P.njobs = (int)K.jobs.size();
        P.launch.inside.lanes = kWave;
        P.depth_cap = wide_depth_cap(K.st);
        P.status = K.checks ? ctx->rec_status.as<unsigned>() : nullptr;
        const long long all = (long long)ctx->cu_count * ctx->batch_blocks_per_cu;
        long long blocks = ncls == 1 ? all : (long long)((double)all * ((double)K.samples / (double)samples) + 0.5);
        const long long need = ((long long)K.total + 255) / 256;
        if (blocks > need) blocks = need;
        if (blocks < 1) blocks = 1;
#define PT_BATCH(ST, HALF_) \
    hipLaunchKernelGGL((k_render_lanes<ST, false, true, true, HALF_>), dim3((unsigned)blocks), dim3(256), 0, s, P)
        if (half) {
            if (K.st == 32) PT_BATCH(32, true);
            else if (K.st == 48) PT_BATCH(48, true);
            else PT_BATCH(64, true);
        } else {
            if (K.st == 32) PT_BATCH(32, false);
            else if (K.st == 48) PT_BATCH(48, false);
            else PT_BATCH(64, false);
        }
#undef PT_BATCH
        PT_HIP(hipGetLastError());
        if (k > 0) {
            PT_HIP(hipEventRecord(ch.join, s));
            PT_HIP(hipStreamWaitEvent(stream, ch.join, 0));
        }
    }
    return PTGPU_OK;
}
}  // namespace ptgpu

extern "C" {

int ptgpu_trace_closest(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const Shape *d_shapes,
                        unsigned int shapeCnt, const Ray *d_rays, int n, float *d_t, int *d_id) {
    PT_CHECK(ctx && d_shapes && d_rays && d_t && d_id, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(shapeCnt >= 1 && n >= 0, PTGPU_ERR_INVALID, "bad sizes");
    PT_HIP(hipSetDevice(ctx->device));
    DevAccel acc;
    PT_TRY(resolve_accel(ctx, bvh, kd, d_shapes, shapeCnt, &acc, true));
    return launch_trace(ctx, acc, shapeCnt, d_rays, nullptr, n, d_t, d_id, nullptr, false);
}

int ptgpu_trace_any(ptgpu_ctx *ctx, ptgpu_clbvh *bvh, ptgpu_kdtree *kd, const Shape *d_shapes, unsigned int shapeCnt,
                    const Ray *d_rays, const float *d_maxt, int n, int *d_hit) {
    PT_CHECK(ctx && d_shapes && d_rays && d_maxt && d_hit, PTGPU_ERR_INVALID, "null argument");
    PT_CHECK(shapeCnt >= 1 && n >= 0, PTGPU_ERR_INVALID, "bad sizes");
    PT_HIP(hipSetDevice(ctx->device));
    DevAccel acc;
    PT_TRY(resolve_accel(ctx, bvh, kd, d_shapes, shapeCnt, &acc, true));
    return launch_trace(ctx, acc, shapeCnt, d_rays, d_maxt, n, nullptr, nullptr, d_hit, true);
}

}  // extern "C"
