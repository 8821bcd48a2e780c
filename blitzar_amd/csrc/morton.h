// Morton key of a position in the root frame (see k_keys.hip for the reference
// behaviour it follows).
#pragma once

#include "bh_internal.h"

namespace bh {

__device__ inline unsigned long long spread21(unsigned int v)
{
    unsigned long long x = v & 0x1fffffu;
    x = (x | (x << 32)) & 0x001f00000000ffffull;
    x = (x | (x << 16)) & 0x001f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

// The reference interleave as it executes: 32-bit lanes, 10-bit masks.
__device__ inline unsigned long long spread_ref32(unsigned int v)
{
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return static_cast<unsigned long long>(v);
}

__device__ inline unsigned int quantise(float p, float lo, float inv)
{
    const float t = fminf(fmaxf((p - lo) * inv, 0.0f), 1.0f);
    const unsigned int q = static_cast<unsigned int>(__fmaf_rn(t, 2097151.0f, 0.5f));
    return min(kQMax, q);
}

// MODE 0: all 21 bits per axis (63-bit key); 1: the reference's 30-bit key.
template <int MODE>
__device__ inline unsigned long long morton_key(double x, double y, double z,
                                                const RootGeom* __restrict__ g)
{
    const unsigned int qx = quantise(static_cast<float>(x), g->lo[0], g->inv[0]);
    const unsigned int qy = quantise(static_cast<float>(y), g->lo[1], g->inv[1]);
    const unsigned int qz = quantise(static_cast<float>(z), g->lo[2], g->inv[2]);
    if (MODE == 1)
        return (spread_ref32(qx) << 2) | (spread_ref32(qy) << 1) | spread_ref32(qz);
    return (spread21(qx) << 2) | (spread21(qy) << 1) | spread21(qz);
}

}  // namespace bh
