// half_bounds.hpp -- binary16 bounds: rounding outward, and whether they blur a tree.
#pragma once

#include "device_util.hpp"

namespace ptgpu {

// binary16 bounds rounded outward: the nearest binary16 (round to nearest even), stepped one
// binary16 ulp down (lo) or up (hi) when it lies on the wrong side of x.  A NaN bound becomes the
// infinity on its own side; values beyond the binary16 range round to +-65504 or the infinity.
__device__ __forceinline__ unsigned short half_down(float x) {
    if (x != x) return 0xFC00u;   // -inf
    const _Float16 h = (_Float16)x;
    unsigned short b = __builtin_bit_cast(unsigned short, h);
    if ((float)h > x) {
        if (b == 0x0000u || b == 0x8000u) b = 0x8001u;   // +-0 -> the largest negative subnormal
        else if (b & 0x8000u) b = (unsigned short)(b + 1u);   // negative: away from zero
        else b = (unsigned short)(b - 1u);                    // positive: toward zero
    }
    return b;
}
__device__ __forceinline__ unsigned short half_up(float x) {
    if (x != x) return 0x7C00u;   // +inf
    const _Float16 h = (_Float16)x;
    unsigned short b = __builtin_bit_cast(unsigned short, h);
    if ((float)h < x) {
        if (b == 0x0000u || b == 0x8000u) b = 0x0001u;   // +-0 -> the smallest positive subnormal
        else if (b & 0x8000u) b = (unsigned short)(b - 1u);   // negative: toward zero
        else b = (unsigned short)(b + 1u);                    // positive: away from zero
    }
    return b;
}

// Do binary16 bounds blur this tree?  They are absolute, so a scene far from the origin (or past 65,504) has
// boxes a binary16 step wide, whatever its shapes' size, and a walk of them visits much of the tree.  Each lane
// widens the leaf boxes of one node, spread evenly over the tree, and the wave compares the areas' sums.  At a sum over four times the exact one the walks of binary16
// and binary32 boxes cost alike (100,000 rays; the scene moved by 16: 1,002-shape soup 67 us here against 71 over binary
// nodes, 327,692-shape mesh 413 against 236; by 256: 256 against 73 us, 146 against 0.24 ms; a 256x256 frame of a
// 20,002-shape soup moved by 16, binary16 / binary32 four-wide nodes: 0.73 / 0.69 ms, by 256: 21.2 / 0.75).
struct BlurSums {
    float exact = 0.f, wide = 0.f;
    __device__ __forceinline__ void add(float x0, float y0, float z0, float x1, float y1, float z1) {
        auto area = [](float dx, float dy, float dz) { return dx * dy + dy * dz + dz * dx; };
        auto lo = [](float v) { return (float)__builtin_bit_cast(_Float16, half_down(v)); };
        auto hi = [](float v) { return (float)__builtin_bit_cast(_Float16, half_up(v)); };
        exact += area(x1 - x0, y1 - y0, z1 - z0);
        wide += area(hi(x1) - lo(x0), hi(y1) - lo(y0), hi(z1) - lo(z0));
    }
};
__host__ __device__ inline bool blurred(float exact, float wide) { return wide > 4.f * exact; }
// of a wave's sums
__device__ __forceinline__ bool half_blurs(BlurSums s) {
    for (int x = 1; x < kWave; x <<= 1) {
        s.exact += __shfl_xor(s.exact, x);
        s.wide += __shfl_xor(s.wide, x);
    }
    return blurred(s.exact, s.wide);
}
// by one wave
__device__ __forceinline__ bool half_blurs(const TNode *nodes, int nnodes) {
    BlurSums s;
    if (nnodes > 0) {
        const TNode t = nodes[(int)((long long)__lane_id() * nnodes / kWave)];
        if (t.r.x < 0 && t.r.x != kEmptyRef) s.add(t.a.x, t.a.y, t.a.z, t.a.w, t.b.x, t.b.y);
        if (t.r.y < 0 && t.r.y != kEmptyRef) s.add(t.b.z, t.b.w, t.c.x, t.c.y, t.c.z, t.c.w);
    }
    return half_blurs(s);
}

}  // namespace ptgpu
