// lbvh_device.hpp -- device bodies of the LBVH build stages.  Each body takes the block index it
// plays and the block count of its scene, so the same code runs as a single-scene kernel (block =
// blockIdx.x) and inside the batched kernels, which map a launch's blocks onto many scenes.
#pragma once

#include <cfloat>

#include "device_util.hpp"
#include "lbvh.hpp"

namespace ptgpu {

__device__ __forceinline__ float shape_f(const Shape *s, int word) {
    return reinterpret_cast<const float *>(s)[word];
}
__device__ __forceinline__ int shape_i(const Shape *s, int word) {
    return reinterpret_cast<const int *>(s)[word];
}

// CLBVH::getBound CLBVH.cpp:49-75 from the Shape words (type @0, p1..p3 / rad,p @1..9).
__device__ __forceinline__ Bound bound_of_words(const float *w, int *type_out) {
    int type = __float_as_int(w[0]);
    *type_out = type;
    Bound b;
    if (type == SPHERE) {
        float rad = w[1], px = w[2], py = w[3], pz = w[4];
        b.min_x = px - rad; b.max_x = px + rad;
        b.min_y = py - rad; b.max_y = py + rad;
        b.min_z = pz - rad; b.max_z = pz + rad;
    } else {
        float x1 = w[1], y1 = w[2], z1 = w[3], x2 = w[4], y2 = w[5], z2 = w[6], x3 = w[7], y3 = w[8], z3 = w[9];
        b.min_x = sel_min(sel_min(x1, x2), x3); b.max_x = sel_max(sel_max(x1, x2), x3);
        b.min_y = sel_min(sel_min(y1, y2), y3); b.max_y = sel_max(sel_max(y1, y2), y3);
        b.min_z = sel_min(sel_min(z1, z2), z3); b.max_z = sel_max(sel_max(z1, z2), z3);
    }
    return b;
}
__device__ __forceinline__ Bound shape_bound(const Shape *s, int *type_out) {
    return bound_of_words(reinterpret_cast<const float *>(s), type_out);
}

// -------------------------------------------------------------------------------------------
// Stage 1: AABBs, scene centroid bounds, Morton codes (CLBVH.cpp:90-164)
// -------------------------------------------------------------------------------------------
constexpr int kBoundsThreads = 256;

__device__ __forceinline__ void reduce6(float *v, float *sh /*6*kBoundsThreads*/) {
    const int tid = threadIdx.x;
    for (int k = 0; k < 6; k++) sh[k * kBoundsThreads + tid] = v[k];
    __syncthreads();
    for (int s = kBoundsThreads / 2; s > 0; s >>= 1) {
        if (tid < s) {
            for (int k = 0; k < 6; k++) {
                float a = sh[k * kBoundsThreads + tid], b = sh[k * kBoundsThreads + tid + s];
                sh[k * kBoundsThreads + tid] = (k & 1) ? sel_max(a, b) : sel_min(a, b);
            }
        }
        __syncthreads();
    }
    for (int k = 0; k < 6; k++) v[k] = sh[k * kBoundsThreads];
}

// Per shape: bound -> Shape.b, index -> Shape.index, centroid; block partial of the centroid
// min/max (max starts at FLT_MIN as CLBVH.cpp:92-96 does) -> partials[bid].
// (block `bid` of `nblocks` working on one scene; the kernels map blocks to scenes)
// A shape's box record, 64 aligned bytes in input order: words 0-9 of the Shape (type, then the
// triangle's vertices or the sphere's radius and centre) and its AABB (min_x, max_x, min_y, max_y,
// min_z, max_z).  The Morton pass reads it instead of the 104-byte Shape and the leaf refit gathers
// it (one aligned 64-byte record per leaf instead of a whole Shape).
struct alignas(16) ShapeBox {
    float4 q[4];
};
static_assert(sizeof(ShapeBox) == 64, "ShapeBox");
__device__ __forceinline__ const float *box_words(const ShapeBox &r) { return reinterpret_cast<const float *>(&r); }

// Contiguous runs of fixed-size records moved between global memory and a wave's LDS staging area
// with 16-byte accesses: lane l's record occupies dwords [l * WORDS, (l + 1) * WORDS) of the stage,
// and the run of `count` (<= 64) records starts at a 16-byte aligned address.  A wave then reads or
// writes its run in WORDS / 4 instructions instead of WORDS dword accesses per lane at a WORDS * 4-byte
// stride (each of which touches as many cache lines as the run does).
template <int WORDS>
__device__ __forceinline__ void wave_store_records(const unsigned *stage, unsigned *dst, int count, int lane) {
    const int total = count * WORDS;
    const int full = total >> 2;
    for (int c = lane; c < full; c += kWave)
        *reinterpret_cast<uint4 *>(dst + 4 * c) = *reinterpret_cast<const uint4 *>(stage + 4 * c);
    const int rem = total - 4 * full;
    if (lane < rem) dst[4 * full + lane] = stage[4 * full + lane];
}
// words [w0, w1) of the stage
__device__ __forceinline__ void wave_store_words(const unsigned *stage, unsigned *dst, int w0, int w1, int lane) {
    for (int c = (w0 >> 2) + lane; 4 * c < w1; c += kWave) {
        if (4 * c >= w0 && 4 * c + 4 <= w1) {
            *reinterpret_cast<uint4 *>(dst + 4 * c) = *reinterpret_cast<const uint4 *>(stage + 4 * c);
        } else {
            for (int e = 4 * c; e < 4 * c + 4; e++)
                if (e >= w0 && e < w1) dst[e] = stage[e];
        }
    }
}
template <int WORDS>
__device__ __forceinline__ void wave_load_records(const unsigned *src, unsigned *stage, int count, int lane) {
    const int total = count * WORDS;
    const int full = total >> 2;
    for (int c = lane; c < full; c += kWave)
        *reinterpret_cast<uint4 *>(stage + 4 * c) = *reinterpret_cast<const uint4 *>(src + 4 * c);
    const int rem = total - 4 * full;
    if (lane < rem) stage[4 * full + lane] = src[4 * full + lane];
}

__device__ __forceinline__ void bounds_body(const Shape *shapes, int n, float *partials, ShapeBox *boxes, int bid,
                                            int nblocks) {
    __shared__ float sh[6 * kBoundsThreads];
    float acc[6] = {FLT_MAX, FLT_MIN, FLT_MAX, FLT_MIN, FLT_MAX, FLT_MIN};
    for (int i = bid * blockDim.x + threadIdx.x; i < n; i += nblocks * blockDim.x) {
        const Shape *s = shapes + i;
        int type;
        Bound b = shape_bound(s, &type);
        const float *wf = reinterpret_cast<const float *>(s);
        ShapeBox r;
        r.q[0] = make_float4(wf[0], wf[1], wf[2], wf[3]);
        r.q[1] = make_float4(wf[4], wf[5], wf[6], wf[7]);
        r.q[2] = make_float4(wf[8], wf[9], b.min_x, b.max_x);
        r.q[3] = make_float4(b.min_y, b.max_y, b.min_z, b.max_z);
        boxes[i] = r;
        float px, py, pz;
        if (type == SPHERE) {
            px = wf[2]; py = wf[3]; pz = wf[4];
        } else {
            px = (b.min_x + b.max_x) / 2.0f;
            py = (b.min_y + b.max_y) / 2.0f;
            pz = (b.min_z + b.max_z) / 2.0f;
        }
        if (px < acc[0]) acc[0] = px;
        if (px > acc[1]) acc[1] = px;
        if (py < acc[2]) acc[2] = py;
        if (py > acc[3]) acc[3] = py;
        if (pz < acc[4]) acc[4] = pz;
        if (pz > acc[5]) acc[5] = pz;
    }
    reduce6(acc, sh);
    if (threadIdx.x < 6) partials[bid * 6 + threadIdx.x] = acc[threadIdx.x];
}

// One block folds a scene's block partials into scene6 = {min_x, max_x, min_y, max_y, min_z, max_z}.
// A separate launch rather than a last-block hand-off: on gfx950 a device-scope release per block
// writes back the L2, which holds every Shape.b just written.
__device__ __forceinline__ void bounds_final_body(const float *partials, int nblocks, float *scene6) {
    __shared__ float sh[6 * kBoundsThreads];
    float fin[6] = {FLT_MAX, FLT_MIN, FLT_MAX, FLT_MIN, FLT_MAX, FLT_MIN};
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x)
        for (int k = 0; k < 6; k++) {
            const float v = partials[b * 6 + k];
            fin[k] = (k & 1) ? sel_max(fin[k], v) : sel_min(fin[k], v);
        }
    reduce6(fin, sh);
    if (threadIdx.x < 6) scene6[threadIdx.x] = fin[threadIdx.x];
}

__device__ __forceinline__ unsigned f2u_code(float v) { return v >= 0.f ? (unsigned)v : 0u; }

__device__ __forceinline__ unsigned expand10(unsigned x) {
    x &= 0x3FFu;
    x = (x | (x << 16)) & 0x030000FFu;
    x = (x | (x << 8)) & 0x0300F00Fu;
    x = (x | (x << 4)) & 0x030C30C3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// CLBVH.cpp:125-164: quantise each centroid to 10 bits per axis (1024 wraps to 0 through the
// low-10-bit interleave) and interleave x above y above z.  The Morton pass also emits the sort key
// ~code (30 bits), so that an ascending stable sort yields the reference's stable descending order,
// and stores the reference's per-shape outputs: index @68, morton_code @72, b @76.
__device__ __forceinline__ unsigned morton_code_of(float px, float py, float pz, const float *scene6) {
    const float mnx = scene6[0], mxx = scene6[1], mny = scene6[2], mxy = scene6[3], mnz = scene6[4],
                mxz = scene6[5];
    unsigned a = f2u_code(((px - mnx) / (mxx - mnx)) * 1024.f);
    unsigned b = f2u_code(((py - mny) / (mxy - mny)) * 1024.f);
    unsigned c = f2u_code(((pz - mnz) / (mxz - mnz)) * 1024.f);
    return (expand10(a) << 2) | (expand10(b) << 1) | expand10(c);
}

// A wave handles 64 consecutive shapes.  When the Shape array is 16-byte aligned, the wave loads its
// 64 whole records (26 words each) into LDS with 16-byte loads, fills in index, morton_code and b,
// and stores the records back whole: full cache lines, where writing only each record's 32-byte tail
// at a 104-byte stride left every line partly written.  The centroid then comes from the record's
// own words; otherwise (a caller's unaligned array) each lane reads its box record and stores its tail.
__device__ __forceinline__ void morton_body(Shape *shapes, int n, const float *scene6, unsigned *keys,
                                            const ShapeBox *boxes, int bid) {
    constexpr int kW = 26;   // words per Shape
    __shared__ __align__(16) unsigned stage[kBoundsThreads / kWave][kWave * kW];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const long long first = (long long)bid * blockDim.x + (long long)wv * kWave;
    if (first >= n) return;   // the whole wave is past the end
    const int count = (long long)n - first < kWave ? (int)((long long)n - first) : kWave;
    const int i = (int)first + lane;
    if ((reinterpret_cast<size_t>(shapes) & 15) == 0) {
        unsigned *st = stage[wv];
        wave_load_records<kW>(reinterpret_cast<const unsigned *>(shapes + first), st, count, lane);
        __builtin_amdgcn_wave_barrier();
        if (lane < count) {
            unsigned *rw = st + lane * kW;
            float w[10];
#pragma unroll
            for (int f = 0; f < 10; f++) w[f] = __uint_as_float(rw[f]);
            int type;
            const Bound b = bound_of_words(w, &type);
            float px, py, pz;
            if (type == SPHERE) {
                px = w[2]; py = w[3]; pz = w[4];
            } else {
                px = (b.min_x + b.max_x) / 2.0f;
                py = (b.min_y + b.max_y) / 2.0f;
                pz = (b.min_z + b.max_z) / 2.0f;
            }
            const unsigned code = morton_code_of(px, py, pz, scene6);
            rw[17] = (unsigned)i;   // index @68
            rw[18] = code;          // morton_code @72
            rw[19] = __float_as_uint(b.min_x); rw[20] = __float_as_uint(b.max_x);   // b @76
            rw[21] = __float_as_uint(b.min_y); rw[22] = __float_as_uint(b.max_y);
            rw[23] = __float_as_uint(b.min_z); rw[24] = __float_as_uint(b.max_z);
            keys[i] = (~code) & 0x3FFFFFFFu;
        }
        __builtin_amdgcn_wave_barrier();
        wave_store_records<kW>(st, reinterpret_cast<unsigned *>(shapes + first), count, lane);
        return;
    }
    if (lane >= count) return;
    const ShapeBox r = boxes[i];
    const float *w = box_words(r);   // w[10..15]: the AABB
    const int type = __float_as_int(w[0]);
    float px, py, pz;
    if (type == SPHERE) {
        px = w[2]; py = w[3]; pz = w[4];
    } else {
        px = (w[10] + w[11]) / 2.0f;
        py = (w[12] + w[13]) / 2.0f;
        pz = (w[14] + w[15]) / 2.0f;
    }
    const unsigned code = morton_code_of(px, py, pz, scene6);
    unsigned *ws = reinterpret_cast<unsigned *>(shapes + i);
    ws[17] = (unsigned)i;   // index @68
    ws[18] = code;          // morton_code @72
    for (int f = 0; f < 6; f++) ws[19 + f] = __float_as_uint(w[10 + f]);   // b @76
    keys[i] = (~code) & 0x3FFFFFFFu;
}

// -------------------------------------------------------------------------------------------
// Stage 2: onesweep LSD radix sort (Adinets & Merrill 2022) for wave64.
//   k_sort_hist:   one read of the keys builds the digit histograms of every pass.
//   k_sort_pass:   per 4096-key tile: the pass's digit bases from its histogram, wave-level match ranking in input order (stable), tile
//                  histogram, decoupled look-back over earlier tiles per digit, LDS shuffle into
//                  digit order, coalesced scatter.  Tile ids come from an atomic counter so every
//                  tile a block waits on has already started.
// -------------------------------------------------------------------------------------------
constexpr int kSortThreads = 256;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr unsigned kFlagAgg = 1u << 30, kFlagPrefix = 2u << 30, kValMask = (1u << 30) - 1;
constexpr unsigned kSpinLimit = 1u << 26;
constexpr int kLookback = 8;   // predecessor status words per look-back round

template <int BITS> struct SortCfg {
    static constexpr int kRadix = 1 << BITS;
    static constexpr unsigned kMask = (unsigned)kRadix - 1;
    static constexpr int kPasses = (30 + BITS - 1) / BITS;
};

template <int BITS>
__device__ __forceinline__ void sort_hist_body(const unsigned *keys, int n, unsigned *hist, int bid, int nblocks) {
    using C = SortCfg<BITS>;
    __shared__ unsigned sh[C::kPasses * C::kRadix];
    for (int j = threadIdx.x; j < C::kPasses * C::kRadix; j += kSortThreads) sh[j] = 0;
    __syncthreads();
    const long long stride = (long long)nblocks * kSortThreads;
    for (long long i = (long long)bid * kSortThreads + threadIdx.x; i < n; i += 4 * stride) {
        unsigned k[4];   // four keys' loads together
#pragma unroll
        for (int j = 0; j < 4; j++) k[j] = i + j * stride < n ? keys[i + j * stride] : 0u;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (i + j * stride >= n) break;
#pragma unroll
            for (int p = 0; p < C::kPasses; p++) atomicAdd(&sh[p * C::kRadix + ((k[j] >> (p * BITS)) & C::kMask)], 1u);
        }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < C::kPasses * C::kRadix; j += kSortThreads)
        if (sh[j]) atomicAdd(&hist[j], sh[j]);
}

// exclusive scan of `v` across the 256 threads of a block; returns the exclusive prefix
__device__ __forceinline__ unsigned block_exscan256(unsigned v, unsigned *s_w, unsigned *total) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    unsigned x = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        unsigned y = __shfl_up(x, o, kWave);
        if (lane >= o) x += y;
    }
    if (lane == kWave - 1) s_w[w] = x;
    __syncthreads();
    unsigned pre = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kSortWaves; k++) {
        unsigned t = s_w[k];
        if (k < w) pre += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return pre + x - v;
}

// The element forms of a pass's input and output.  kSplit: a key array and a value array (an input
// without a value array takes each element's index as its value).  kPacked: one 8-byte word per
// element, the key in its low half and the value in its high half, read from / written to the
// keys_in / keys_out pointer (vals_in / vals_out unused): one load and one store per element, and each
// tile's digit runs are twice as long in bytes as in either split array, so the scatter leaves fewer
// partly written cache lines.
enum SortForm { kSplit = 0, kPacked = 1 };

template <int BITS, int IN = kSplit, int OUT = kSplit>
__device__ __forceinline__ void sort_pass_body(const unsigned *__restrict__ keys_in, const unsigned *__restrict__ vals_in,
                                               unsigned *__restrict__ keys_out, unsigned *__restrict__ vals_out, int n,
                                               int shift, const unsigned *__restrict__ digit_count, unsigned *status,
                                               unsigned tile, unsigned *err) {
    using C = SortCfg<BITS>;
    __shared__ unsigned long long s_kv[kSortTile];   // the tile in digit order, key | value << 32
    __shared__ unsigned s_wcnt[kSortWaves][C::kRadix];
    __shared__ unsigned s_lofs[C::kRadix];
    __shared__ unsigned s_gofs[C::kRadix];
    __shared__ unsigned s_w[kSortWaves];

    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
    for (int j = tid; j < kSortWaves * C::kRadix; j += kSortThreads) (&s_wcnt[0][0])[j] = 0;
    __syncthreads();
    const long long base = (long long)tile * kSortTile;
    const long long wbase = base + (long long)w * kWave * kSortItems;

    unsigned k[kSortItems], v[kSortItems], rank[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        long long idx = wbase + j * kWave + lane;
        bool valid = idx < n;
        if (IN == kPacked) {
            const unsigned long long x = valid ? reinterpret_cast<const unsigned long long *>(keys_in)[idx] : ~0ull;
            k[j] = (unsigned)x;
            v[j] = (unsigned)(x >> 32);
        } else {
            k[j] = valid ? keys_in[idx] : 0xFFFFFFFFu;
            v[j] = valid ? (vals_in ? vals_in[idx] : (unsigned)idx) : 0u;
        }
    }
    const unsigned long long lt = lanemask_lt();
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        long long idx = wbase + j * kWave + lane;
        bool valid = idx < n;
        unsigned digit = (k[j] >> shift) & C::kMask;
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < BITS; b++) {
            bool bit = (digit >> b) & 1u;
            unsigned long long m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        unsigned pre = 0;
        if (valid) pre = s_wcnt[w][digit];
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            rank[j] = pre + (unsigned)__popcll(peers & lt);
            if ((peers & lt) == 0) s_wcnt[w][digit] = pre + (unsigned)__popcll(peers);
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // per digit: wave-exclusive offsets, tile count, tile-local offsets, global base (look-back)
    for (int d0 = 0; d0 < C::kRadix; d0 += kSortThreads) {
        const int d = d0 + tid;
        unsigned cnt = 0;
        if (d < C::kRadix) {
            unsigned run = 0;
#pragma unroll
            for (int q = 0; q < kSortWaves; q++) {
                unsigned c = s_wcnt[q][d];
                s_wcnt[q][d] = run;
                run += c;
            }
            cnt = run;
        }
        unsigned tot;
        const unsigned dbase = block_exscan256(d < C::kRadix ? digit_count[d] : 0u, s_w, &tot);   // kRadix <= 256
        unsigned lofs = block_exscan256(cnt, s_w, &tot);
        if (d < C::kRadix) {
            s_lofs[d] = lofs;
            unsigned *my = status + (size_t)tile * C::kRadix + d;
            unsigned prefix = 0;
            if (tile == 0) {
                st_relaxed(my, kFlagPrefix | cnt);
            } else {
                st_relaxed(my, kFlagAgg | cnt);
                // Windowed look-back: the status words of kLookback predecessors are loaded together
                // and summed nearest first up to the first inclusive prefix, so a walk over tiles
                // that have published only their counts costs one round trip per window instead of
                // one per tile.  A word not yet published stops the window; the walk resumes there.
                long long t = (long long)tile - 1;
                unsigned spins = 0;
                while (t >= 0) {
                    unsigned w[kLookback];
#pragma unroll
                    for (int k = 0; k < kLookback; k++)
                        w[k] = t - k >= 0 ? ld_relaxed(status + (size_t)(t - k) * C::kRadix + d) : kFlagPrefix;
                    bool stop = false, found = false;
                    int adv = 0;
#pragma unroll
                    for (int k = 0; k < kLookback; k++) {
                        if (stop) continue;
                        const unsigned flag = w[k] & ~kValMask;
                        if (flag == 0) {
                            stop = true;
                        } else {
                            prefix += w[k] & kValMask;
                            adv++;
                            if (flag == kFlagPrefix) stop = found = true;
                        }
                    }
                    if (found) break;
                    t -= adv;
                    if (adv < kLookback && ++spins > kSpinLimit) { atomicOr(err, 1u); break; }
                }
                st_relaxed(my, kFlagPrefix | ((prefix + cnt) & kValMask));
            }
            s_gofs[d] = dbase + prefix;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        long long idx = wbase + j * kWave + lane;
        if (idx < n) {
            unsigned digit = (k[j] >> shift) & C::kMask;
            unsigned lpos = s_lofs[digit] + s_wcnt[w][digit] + rank[j];
            s_kv[lpos] = (unsigned long long)k[j] | ((unsigned long long)v[j] << 32);
        }
    }
    __syncthreads();
    long long rem = (long long)n - base;
    const int count = rem < kSortTile ? (int)rem : kSortTile;
    for (int i = tid; i < count; i += kSortThreads) {
        const unsigned long long x = s_kv[i];
        unsigned key = (unsigned)x;
        unsigned digit = (key >> shift) & C::kMask;
        unsigned dest = s_gofs[digit] + (unsigned)i - s_lofs[digit];
        if (OUT == kPacked) {
            reinterpret_cast<unsigned long long *>(keys_out)[dest] = x;
        } else {
            keys_out[dest] = key;
            vals_out[dest] = (unsigned)(x >> 32);
        }
    }
}

// -------------------------------------------------------------------------------------------
// Stage 3: Karras radix tree over leaf indices (BVH.cl:127-208).  The prefix length of two leaves
// is clz(i ^ j); the tree is therefore the binary radix tree of 0..N-1.
// -------------------------------------------------------------------------------------------
__device__ __forceinline__ int delta_idx(int i, int j, int n) {
    return (j >= 0 && j < n) ? __clz(i ^ j) : -1;
}

// Each thread also writes the reference's initial contents (CLBVH.cpp:83-88: internal nodes zeroed,
// leaves filled with 0xFF bytes) into every field of internal node i and leaf i but nParent, which
// the parent's thread writes (the root's is 0); thread n-2 fills leaf n-1 as well.  One pass of
// whole records instead of two fills followed by scattered field stores.
__device__ __forceinline__ void fill_leaf_record(BVHNodeGPU *l) {
    int *w = reinterpret_cast<int *>(l);
    for (int f = 0; f < 15; f++)
        if (f != 6) w[f] = -1;   // nParent (field 6) comes from the parent
}

__device__ __forceinline__ void karras_body(int n, BVHNodeGPU *btn, BVHNodeGPU *btl, int bid) {
    const int i = bid * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    fill_leaf_record(btl + i);
    if (i == n - 2) fill_leaf_record(btl + n - 1);
    const int d = (delta_idx(i, i + 1, n) - delta_idx(i, i - 1, n)) > 0 ? 1 : -1;
    const int dmin = delta_idx(i, i - d, n);
    int lmax = 2;
    while (delta_idx(i, i + lmax * d, n) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta_idx(i, i + (l + t) * d, n) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta_idx(i, j, n);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta_idx(i, i + (s + t) * d, n) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * d + (d < 0 ? d : 0);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    int leafflag = 0;
    if (lo == gamma) { leafflag = 2; btl[gamma].nParent = i; }
    else btn[gamma].nParent = i;
    if (hi == gamma + 1) { leafflag = 2; btl[gamma + 1].nParent = i; }
    else btn[gamma + 1].nParent = i;
    int *w = reinterpret_cast<int *>(btn + i);
    w[0] = lo;           // min
    w[1] = hi;           // max
    w[2] = 0;            // nShape
    w[3] = leafflag;     // leaf
    w[4] = gamma;        // nLeft
    w[5] = gamma + 1;    // nRight
    if (i == 0) w[6] = 0;   // the root's nParent
    for (int f = 7; f < 15; f++) w[f] = 0;   // bound, cost, area
}

// -------------------------------------------------------------------------------------------
// Stage 4: leaves + bottom-up refit (BVH.cl:214-258).  Leaf k takes the AABB and index of shape
// sorted[k]; a parent's bound is the merge of its (left, right) child bounds, where a child is a
// leaf iff nLeft == min / nRight == max.  Also writes the traversal layout (TNode per internal
// node, Prim per leaf).
// -------------------------------------------------------------------------------------------
// w: words 0-9 of a Shape (a ShapeBox's first ten)
__device__ __forceinline__ Prim make_prim(const float *w, int id) {
    const int type = __float_as_int(w[0]) | kLastInLeaf;   // one primitive per leaf
    Prim p;
    if ((type & 0xff) == SPHERE) {
        p.p0 = make_float4(w[2], w[3], w[4], __int_as_float(id));
        p.p1 = make_float4(w[1], 0.f, 0.f, __int_as_float(type));
        p.p2 = make_float4(0.f, 0.f, 0.f, __int_as_float(type));
    } else {
        float x1 = w[1], y1 = w[2], z1 = w[3];
        p.p0 = make_float4(x1, y1, z1, __int_as_float(id));
        p.p1 = make_float4(w[4] - x1, w[5] - y1, w[6] - z1, __int_as_float(type));
        p.p2 = make_float4(w[7] - x1, w[8] - y1, w[9] - z1, __int_as_float(type));
    }
    return p;
}

__device__ __forceinline__ void store_bound(BVHNodeGPU *node, const Bound &b) {
    float *f = reinterpret_cast<float *>(&node->bound);
    f[0] = b.min_x; f[1] = b.max_x; f[2] = b.min_y; f[3] = b.max_y; f[4] = b.min_z; f[5] = b.max_z;
}

__device__ __forceinline__ TNode make_tnode(const Bound &L, const Bound &R, int rl, int rr, int cl, int cr) {
    TNode t;
    t.a = make_float4(L.min_x, L.min_y, L.min_z, L.max_x);
    t.b = make_float4(L.max_y, L.max_z, R.min_x, R.min_y);
    t.c = make_float4(R.min_z, R.max_x, R.max_y, R.max_z);
    t.r = make_int4(rl, rr, cl, cr);
    return t;
}

// -------------------------------------------------------------------------------------------
// Stage 4 (index-keyed trees): fence-free refit by level passes.
// The Karras tree over leaf indices is the binary radix tree of 0..N-1, so every internal node
// covers an aligned block [j*2^s, min((j+1)*2^s, N) - 1] of leaves, with s = ceil(log2(len)),
// and its Karras index is a closed form of (lo, hi, N): the node is the LEFT child of its parent
// (index hi) iff bit s of lo is 0 and leaves remain after the block, otherwise it is the right
// child or the root (index lo).  One workgroup reduces 1024 consecutive items (leaves, or subtree
// roots of the previous pass) bottom-up in LDS, merging (left, right) exactly as BVH.cl:112-122,
// writes every internal node's bound and TNode on the way, and hands its block root to the next
// pass.  No atomics, no cross-workgroup visibility, deterministic; identical results to the
// reference's visit-flag refit (BVH.cl:214-258), whose arrival order does not change a bound.
// -------------------------------------------------------------------------------------------
constexpr int kRefitLog = 10;
constexpr int kRefitItems = 1 << kRefitLog;

__device__ __forceinline__ int karras_index(long long lo, long long hi, int n) {
    const int len = (int)(hi - lo + 1);
    const int s = 32 - __clz(len - 1);   // ceil(log2(len)), len >= 2
    return (lo + (1ll << s) <= n - 1 && !((lo >> s) & 1)) ? (int)hi : (int)lo;
}
__device__ __forceinline__ int child_ref(long long lo, long long hi, int n) {
    return lo == hi ? ~(int)lo : karras_index(lo, hi, n);
}
// Parent of the node (or leaf, s = 0) that covers the aligned block of level s starting at lo: the
// first enclosing block whose right half is not empty (a block with an empty right half is the
// same node one level up).  The root's nParent is 0 (the reference zeroes internal nodes), a lone
// leaf's stays 0xFF-filled.
__device__ __forceinline__ int index_tree_parent(long long lo, int s, int n) {
    if (n < 2) return -1;
    for (int t = s + 1; t < 40; t++) {
        const long long plo = lo & ~((1ll << t) - 1);
        const long long pmid = plo + (1ll << (t - 1));
        if (pmid <= (long long)n - 1) {
            const long long phi_full = plo + (1ll << t) - 1;
            return karras_index(plo, phi_full < n - 1 ? phi_full : (long long)n - 1, n);
        }
    }
    return 0;
}
// Whole reference records (BVHNodeGPU.h:4-16, 15 words) in one pass: a leaf keeps the 0xFF fill
// (CLBVH.cpp:83-88) in every field but nShape, nParent and bound; an internal node gets its Karras
// fields (min, max, leaf = 2 when a child is a leaf, nLeft = split, nRight = split + 1, nParent)
// with nShape, cost and area zero.
__device__ __forceinline__ void write_leaf_record(BVHNodeGPU *l, int sid, int parent, const Bound &B) {
    int *w = reinterpret_cast<int *>(l);
    w[0] = -1; w[1] = -1; w[2] = sid; w[3] = -1; w[4] = -1; w[5] = -1; w[6] = parent;
    store_bound(l, B);
    w[13] = -1; w[14] = -1;
}
__device__ __forceinline__ void write_node_record(BVHNodeGPU *d, int lo, int hi, int mid, int parent, const Bound &B) {
    int *w = reinterpret_cast<int *>(d);
    w[0] = lo; w[1] = hi; w[2] = 0; w[3] = (lo == mid - 1 || hi == mid) ? 2 : 0;
    w[4] = mid - 1; w[5] = mid; w[6] = parent;
    store_bound(d, B);
    w[13] = 0; w[14] = 0;
}

template <bool LEAF>
__device__ __forceinline__ void refit_levels_body(const ShapeBox *boxes, const unsigned *sorted, int n, int s0, int levels,
                                                  const float *in_bounds, float *out_bounds, BVHNodeGPU *btn,
                                                  BVHNodeGPU *btl, TNode *tnodes, Prim *prims, bool tnodes_on, int bid) {
    __shared__ float sb[6][kRefitItems];
    // per wave: 64 leaf records (15 words) or 64 Prims (12 words), staged for contiguous stores
    __shared__ __align__(16) unsigned stage[LEAF ? 4 : 1][LEAF ? 64 * 15 : 4];
    const long long item_base = (long long)bid * kRefitItems;
    const long long m = ((long long)n + (1ll << s0) - 1) >> s0;   // items at level s0
    // leaf level: all of this thread's gathers are issued before any store (a store between them
    // would make each gather wait for the stores before it)
    constexpr int kPer = kRefitItems / 256;
    int sids[kPer];
    ShapeBox recs[kPer];
    if (LEAF) {
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const long long it = item_base + threadIdx.x + q * 256;
            sids[q] = it < m ? (int)sorted[it] : -1;
        }
#pragma unroll
        for (int q = 0; q < kPer; q++)
            if (sids[q] >= 0) recs[q] = boxes[sids[q]];
    }
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        const int j = threadIdx.x + q * 256;
        const long long it = item_base + j;
        if (LEAF) {
            // the wave's 64 items are consecutive leaves: their records go out as one contiguous run
            const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
            const long long first = it - lane;
            const int count = first >= m ? 0 : (m - first < kWave ? (int)(m - first) : kWave);
            unsigned *st = stage[wv];
            Bound B;
            const float *w = box_words(recs[q]);
            if (it < m) {
                B.min_x = w[10]; B.max_x = w[11]; B.min_y = w[12]; B.max_y = w[13]; B.min_z = w[14]; B.max_z = w[15];
                BVHNodeGPU rec;
                write_leaf_record(&rec, sids[q], index_tree_parent(it, 0, n), B);
                const unsigned *rw = reinterpret_cast<const unsigned *>(&rec);
#pragma unroll
                for (int f = 0; f < 15; f++) st[lane * 15 + f] = rw[f];
                sb[0][j] = B.min_x; sb[1][j] = B.max_x; sb[2][j] = B.min_y;
                sb[3][j] = B.max_y; sb[4][j] = B.min_z; sb[5][j] = B.max_z;
            }
            __builtin_amdgcn_wave_barrier();
            wave_store_records<15>(st, reinterpret_cast<unsigned *>(btl + first), count, lane);
            __builtin_amdgcn_wave_barrier();
            if (it < m) {
                const Prim p = make_prim(w, sids[q]);
                const unsigned *pw = reinterpret_cast<const unsigned *>(&p);
#pragma unroll
                for (int f = 0; f < 12; f++) st[lane * 12 + f] = pw[f];
            }
            __builtin_amdgcn_wave_barrier();
            wave_store_records<12>(st, reinterpret_cast<unsigned *>(prims + first), count, lane);
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        if (it >= m) continue;
        Bound B;
        {
            const float *f = in_bounds + it * 6;
            B.min_x = f[0]; B.max_x = f[1]; B.min_y = f[2]; B.max_y = f[3]; B.min_z = f[4]; B.max_z = f[5];
        }
        sb[0][j] = B.min_x; sb[1][j] = B.max_x; sb[2][j] = B.min_y;
        sb[3][j] = B.max_y; sb[4][j] = B.min_z; sb[5][j] = B.max_z;
    }
    __syncthreads();
    for (int lev = 1; lev <= levels; lev++) {
        const int s = s0 + lev;
        const int nodes_here = kRefitItems >> lev;
        for (int j = threadIdx.x; j < nodes_here; j += 256) {
            const long long lo = (item_base + ((long long)j << lev)) << s0;
            const long long mid = lo + (1ll << (s - 1));
            if (mid > (long long)n - 1) continue;   // right half empty (or block past the end): collapsed
            const long long hi_full = lo + (1ll << s) - 1;
            const long long hi = hi_full < n - 1 ? hi_full : (long long)n - 1;
            const int ls = j << lev, rs = ls + (1 << (lev - 1));
            Bound L, R;
            L.min_x = sb[0][ls]; L.max_x = sb[1][ls]; L.min_y = sb[2][ls];
            L.max_y = sb[3][ls]; L.min_z = sb[4][ls]; L.max_z = sb[5][ls];
            R.min_x = sb[0][rs]; R.max_x = sb[1][rs]; R.min_y = sb[2][rs];
            R.max_y = sb[3][rs]; R.min_z = sb[4][rs]; R.max_z = sb[5][rs];
            const Bound M = merge_bounds(L, R);
            sb[0][ls] = M.min_x; sb[1][ls] = M.max_x; sb[2][ls] = M.min_y;
            sb[3][ls] = M.max_y; sb[4][ls] = M.min_z; sb[5][ls] = M.max_z;
            const int idx = karras_index(lo, hi, n);
            if (LEAF) {   // kept at the split, which no later level reads, for the records below
                sb[0][rs] = M.min_x; sb[1][rs] = M.max_x; sb[2][rs] = M.min_y;
                sb[3][rs] = M.max_y; sb[4][rs] = M.min_z; sb[5][rs] = M.max_z;
            } else {
                write_node_record(btn + idx, (int)lo, (int)hi, (int)mid, index_tree_parent(lo, s, n), M);
            }
            if (tnodes_on) {
                const int rl = child_ref(lo, mid - 1, n), rr = child_ref(mid, hi, n);
                tnodes[idx] = make_tnode(L, R, rl, rr, rl < 0 ? 1 : 0, rr < 0 ? 1 : 0);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6 && out_bounds) out_bounds[(long long)bid * 6 + threadIdx.x] = sb[threadIdx.x][0];
    if (LEAF) {
        // The block's node records in the order of their indices, a wave's 64 as one contiguous run (as 15 words a
        // lane, 60 bytes apart: 307 us for the pass over 4,000,003 shapes, so: 262).  An odd index is the last
        // leaf of a left child: its trailing ones give the node's level; an even one is the first leaf of any other
        // node.  Nodes that reach out of the block, at most its first and last index, belong to a later pass.
        const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
        unsigned *st = stage[wv];
#pragma unroll 1
        for (int q = 0; q < kPer; q++) {
            const long long first = item_base + (threadIdx.x - lane) + q * 256;
            const int i = (int)(first + lane);
            bool mine = first + lane <= (long long)n - 2;
            if (mine) {
                long long lo, hi;
                if (i & 1) {
                    const int k = __builtin_ctz(~(unsigned)i);
                    lo = (long long)i + 1 - (1ll << k);
                    hi = i;
                } else {
                    lo = i;
                    hi = i ? (long long)i + (1ll << __builtin_ctz((unsigned)i)) - 1 : (long long)n - 1;
                    if (hi > n - 1) hi = n - 1;
                }
                mine = lo >= item_base && hi < item_base + kRefitItems;
                if (mine) {
                    const int s = 32 - __clz((int)(hi - lo));   // ceil(log2(len)), len >= 2
                    const long long mid = lo + (1ll << (s - 1));
                    const int m0 = (int)(mid - item_base);
                    Bound M;
                    M.min_x = sb[0][m0]; M.max_x = sb[1][m0]; M.min_y = sb[2][m0];
                    M.max_y = sb[3][m0]; M.min_z = sb[4][m0]; M.max_z = sb[5][m0];
                    BVHNodeGPU rec;
                    write_node_record(&rec, (int)lo, (int)hi, (int)mid, index_tree_parent(lo, s, n), M);
                    const unsigned *rw = reinterpret_cast<const unsigned *>(&rec);
#pragma unroll
                    for (int f = 0; f < 15; f++) st[lane * 15 + f] = rw[f];
                }
            }
            const unsigned long long have = __ballot(mine);
            __builtin_amdgcn_wave_barrier();
            if (have)
                wave_store_words(st, reinterpret_cast<unsigned *>(btn + first), 15 * (__ffsll((long long)have) - 1),
                                 15 * (64 - __builtin_clzll(have)), lane);
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// -------------------------------------------------------------------------------------------
// Traversal tree: Karras radix tree over the sorted Morton keys (ties broken by leaf index), the
// standard LBVH.  The reference exports the index-keyed tree (kept bit-exact in btn/btl); the
// traversal layout may use any tree over the same leaves, and the Morton-keyed one halves the SAH
// cost of the index-keyed one on the C2 soup (159 vs 318).  Closest-hit and any-hit results do
// not depend on the tree.
// -------------------------------------------------------------------------------------------
__device__ __forceinline__ int delta_key(const unsigned *keys, int i, int j, int n) {
    if (j < 0 || j >= n) return -1;
    const unsigned x = keys[i] ^ keys[j];
    return x ? __clz(x) : 32 + __clz(i ^ j);
}

// Topology and bounds bottom-up, in one pass per level of lists.  An item is a finished subtree: a leaf, or
// what an earlier level left over.  Items stand in leaf order, and between neighbours stands their prefix
// length D.  An item [a, b] belongs under the split with the longer prefix of its two sides: the left child
// of the split after b, or the right child of the split before a (the tree over the adjacent prefixes is
// the radix tree).  The first child to reach a split waits in the split's slot; the second merges both,
// writes the traversal node and goes on with it.  A node's index is the radix tree's: its last leaf where it
// is a left child, its first leaf otherwise.  No topology pass, parent links or counters in memory, and a
// node's children, range and side are known from the items alone.
//
// One wave works a list: 128 leaves, or the leftovers of kMFan lists (which the other waves of its workgroup help to
// load: a workgroup of a single wave with more than 17 KB of LDS was not placed beside a render's workgroups at all,
// wherever they left room, and a build on another stream ended with the render; so a 65,538-shape build beside one of two
// workgroups per CU takes 0.27 ms, not 2 to 6).  Its lanes hold one item each, and a
// lane whose item waits takes the next one, so the wave's steps stay full until its items run out; one
// thread per leaf climbing its parents left most lanes of each wave idle after two steps, and read the
// topology from memory.  What bounds it: the step's instructions and its LDS round trips.  4,000,003 shapes:
// topology, chunk climb and the two climbs above it 907 us; this pass and its upper levels 250 us (512 leaves a list:
// 244 us, but 1,003 shapes 9 us longer: their waves' chains are what counts there).
//
// Leftovers: items whose split is not inside the list, and those that wait for one that is not.  They are
// cut by nodes that span an end of the list, whose prefixes differ: at most one per prefix length and end, so
// 2 * 62 + 1 (30-bit codes, ties split by the index).  More come only of unsorted keys (a failed sort): the
// surplus is dropped and the build's error word set.
constexpr int kMChunk = 128;      // leaves per list of the first level
constexpr int kMFan = 16;         // lists per list of the next level
static_assert((kMFan & (kMFan - 1)) == 0, "an item's list is found by halving");
constexpr int kMThreads = 256;    // of an upper level's workgroups
constexpr int kMItems = 128;      // room for a list's leftovers (at most 125)
constexpr int kMMaxLevels = 8;    // lists of 2^30 leaves: 2^23, then a sixteenth at each level
struct alignas(16) MItem {
    float4 q0;   // bound: min_x, max_x, min_y, max_y
    float2 q1;   // min_z, max_z
    int first;   // first leaf
    int dh;      // bits 0-7: prefix length with the leaf before it, plus one (0 at the tree's start); bits 8-: height
};
static_assert(sizeof(MItem) == 32, "MItem");

template <bool LEAVES>
struct MTreeList {
    static constexpr int kCap = LEAVES ? kMChunk : kMFan * (kMItems - 3);
    float2 b[3][kCap + 1];            // slot s: the bound waiting at the split before item s; item s-1 until it is taken
    unsigned tag[kCap + 1];           // bit 31: an item waits, bit 30: the left child, bits 16-29: height, 0-15: its far end
    int first[LEAVES ? 1 : kCap + 1];
    unsigned char d[kCap + 4];        // d[s]: prefix length across split s, plus one
    unsigned char h[LEAVES ? 4 : kCap + 4];
    unsigned starts[(kCap + 31) / 32];
    int offs[kMFan + 1];
};

// `lists_in`: lists of the level below (upper levels).  out / out_cnt: this level's leftovers.
template <bool LEAVES>
__device__ __forceinline__ void mtree_body(int n, const unsigned *keys, const BVHNodeGPU *btl, const MItem *in,
                                           const int *in_cnt, int lists_in, MItem *out, int *out_cnt, TNode *tnodes,
                                           unsigned *root_height, unsigned *err, int bid) {
    __shared__ MTreeList<LEAVES> S;
    constexpr int kCap = MTreeList<LEAVES>::kCap;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    constexpr int kThreads = LEAVES ? kWave : kMThreads;
    const unsigned long long lt = lanemask_lt();
    const int base = bid * kMChunk;
    int count;
    auto stage = [&](int item, float2 x, float2 y, float2 z) {
        S.b[0][item + 1] = x;
        S.b[1][item + 1] = y;
        S.b[2][item + 1] = z;
    };
    if (LEAVES) {
        count = n - base < kMChunk ? n - base : kMChunk;
#pragma unroll 4
        for (int i = lane; i < count; i += kWave) {
            const float *f = reinterpret_cast<const float *>(&btl[base + i].bound);
            stage(i, make_float2(f[0], f[1]), make_float2(f[2], f[3]), make_float2(f[4], f[5]));
        }
#pragma unroll 4
        for (int i = lane; i <= count; i += kWave) {
            const int k = base + i;
            S.d[i] = (unsigned char)(k < n ? delta_key(keys, k, k - 1, n) + 1 : 0);
        }
    } else {
        const int l0 = bid * kMFan;
        const int lists = lists_in - l0 < kMFan ? lists_in - l0 : kMFan;
        int c = lane < lists ? in_cnt[l0 + lane] : 0;
        c = c < kMItems - 3 ? c : kMItems - 3;
        int run = c;
        for (int x = 1; x < kMFan; x <<= 1) {
            const int o = __shfl_up(run, x);
            if (lane >= x) run += o;
        }
        if (lane < kMFan) S.offs[lane + 1] = run;
        if (lane == 0) S.offs[0] = 0;
        __syncthreads();
        count = S.offs[kMFan];
#pragma unroll 4
        for (int i = tid; i < count; i += kThreads) {
            int q = 0;
            for (int x = kMFan >> 1; x > 0; x >>= 1)
                if (S.offs[q + x] <= i) q += x;
            const MItem m = in[(size_t)(l0 + q) * kMItems + (i - S.offs[q])];
            stage(i, make_float2(m.q0.x, m.q0.y), make_float2(m.q0.z, m.q0.w), m.q1);
            S.first[i] = m.first;
            S.d[i] = (unsigned char)(m.dh & 0xff);
            S.h[i] = (unsigned char)(m.dh >> 8);
        }
        if (tid == 0) {
            const bool more = l0 + kMFan < lists_in;
            const MItem *nx = in + (size_t)(l0 + kMFan) * kMItems;
            S.first[count] = more ? nx->first : n;
            S.d[count] = (unsigned char)(more ? nx->dh & 0xff : 0);
        }
    }
    for (int s = tid; s <= count; s += kThreads) S.tag[s] = 0u;
    for (int s = tid; s < (kCap + 31) / 32; s += kThreads) S.starts[s] = 0u;
    __syncthreads();
    if (tid >= kWave) return;   // one wave from here on: no barriers
    auto first_leaf = [&](int item) { return LEAVES ? base + item : S.first[item]; };

    bool on = false;
    int a = 0, b = 0, h = 0, next = 0;
    float2 bx = make_float2(0.f, 0.f), by = bx, bz = bx;
    for (;;) {
        // lanes without an item take the next ones (a slot's own item is taken before anything waits there)
        if (next < count) {
            const unsigned long long want = __ballot(!on);
            const int k = next + (int)__popcll(want & lt);
            if (!on && k < count) {
                on = true;
                a = b = k;
                h = LEAVES ? 0 : S.h[k];
                bx = S.b[0][k + 1];
                by = S.b[1][k + 1];
                bz = S.b[2][k + 1];
            }
            next += (int)__popcll(want);
        }
        if (!__ballot(on)) break;
        int s = 0;
        bool left = false;
        unsigned other = 0u;
        if (on) {
            const int da = S.d[a], db = S.d[b + 1];
            if ((da | db) == 0) {   // the whole tree
                *root_height = (unsigned)h;
                on = false;
            } else {
                left = db > da;
                s = left ? b + 1 : a;
                other = atomicExch(&S.tag[s], 0x80000000u | (left ? 0x40000000u : 0u) | ((unsigned)h << 16) |
                                                  (unsigned)(left ? a : b));
            }
        }
        // all lanes' arrivals are in (one wave, in order): the first ones' bounds are stored before the second
        // ones read them, also where both come in the same step
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
        if (on && !other) {
            S.b[0][s] = bx;
            S.b[1][s] = by;
            S.b[2][s] = bz;
            on = false;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
        if (on) {
            const float2 ox = S.b[0][s], oy = S.b[1][s], oz = S.b[2][s];
            S.tag[s] = 0u;
            const int far = (int)(other & 0xffffu), oh = (int)((other >> 16) & 0x3fffu);
            Bound L, R;
            L.min_x = left ? bx.x : ox.x; L.max_x = left ? bx.y : ox.y;
            L.min_y = left ? by.x : oy.x; L.max_y = left ? by.y : oy.y;
            L.min_z = left ? bz.x : oz.x; L.max_z = left ? bz.y : oz.y;
            R.min_x = left ? ox.x : bx.x; R.max_x = left ? ox.y : bx.y;
            R.min_y = left ? oy.x : by.x; R.max_y = left ? oy.y : by.y;
            R.min_z = left ? oz.x : bz.x; R.max_z = left ? oz.y : bz.y;
            const Bound M = merge_bounds(L, R);
            bx = make_float2(M.min_x, M.max_x);
            by = make_float2(M.min_y, M.max_y);
            bz = make_float2(M.min_z, M.max_z);
            if (left) b = far; else a = far;
            h = (h > oh ? h : oh) + 1;
            const int lo = first_leaf(a), g = first_leaf(s) - 1, hi = first_leaf(b + 1) - 1;
            const int rl = lo == g ? ~g : g, rr = g + 1 == hi ? ~hi : g + 1;
            const int p = S.d[b + 1] > S.d[a] ? hi : lo;
            if ((unsigned)p < (unsigned)(n - 1)) tnodes[p] = make_tnode(L, R, rl, rr, rl < 0 ? 1 : 0, rr < 0 ? 1 : 0);
        }
    }
    if (!out) return;
    // the items that still wait, in leaf order
    auto start_of = [&](int s, unsigned t) { return t & 0x40000000u ? (int)(t & 0xffffu) : s; };
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
    for (int s = lane; s <= count; s += kWave) {
        const unsigned t = S.tag[s];
        const int a0 = start_of(s, t);
        if (t && a0 < count) atomicOr(&S.starts[a0 >> 5], 1u << (a0 & 31));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
    int total = 0;
    for (int w = 0; w < (kCap + 31) / 32; w++) total += __popc(S.starts[w]);
    if (lane == 0) {
        out_cnt[bid] = total;
        if (total > kMItems - 3) atomicOr(err, 2u);
    }
    MItem *o = out + (size_t)bid * kMItems;
    for (int s = lane; s <= count; s += kWave) {
        const unsigned t = S.tag[s];
        const int a0 = start_of(s, t);
        if (!t || a0 >= count) continue;
        int rank = __popc(S.starts[a0 >> 5] & ((1u << (a0 & 31)) - 1u));
        for (int w = 0; w < (a0 >> 5); w++) rank += __popc(S.starts[w]);
        if (rank >= kMItems - 3) continue;
        MItem m;
        const float2 x = S.b[0][s], y = S.b[1][s];
        m.q0 = make_float4(x.x, x.y, y.x, y.y);
        m.q1 = S.b[2][s];
        m.first = first_leaf(a0);
        m.dh = (int)S.d[a0] | (int)(((t >> 16) & 0x3fffu) << 8);
        o[rank] = m;
    }
}

// Lists of each level over n leaves; their count.
inline int mtree_levels(int n, int *lists) {
    int k = 0;
    lists[0] = (n + kMChunk - 1) / kMChunk;
    while (lists[k] > 1) {
        lists[k + 1] = (lists[k] + kMFan - 1) / kMFan;
        k++;
    }
    return k + 1;
}

}  // namespace ptgpu
