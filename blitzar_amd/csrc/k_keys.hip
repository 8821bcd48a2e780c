// AABB reduction, root geometry and Morton key generation for octree_hip.
//
// Reference behaviour followed:
//   AABB over positions         engine/physics/octree/cuda/linear/OctBuild.inl:58-72
//   key quantisation            engine/physics/octree/cuda/linear/OctKeyKernels.inl:22-46
//   bit interleave              engine/physics/octree/morton/OctMortonCodes.inl:7-22
// The quantisation is the reference's per-axis formula
//   t = clamp((p - lo) * inv, 0, 1),  q = min(2^21-1, (uint)fma(t, 2^21-1, 0.5))
// (nvcc's default --fmad=true contracts the reference's `t * 2097151.0f + 0.5f`
// into that FMA). Key mode 0 interleaves all 21 bits per axis (63-bit key);
// key mode 1 reproduces the reference's interleave, which runs on 32-bit lanes
// with the 10-bit masks and therefore keeps only the low 10 bits per axis.
//
// HBM traffic: AABB reads 24 B/particle (FP64 SoA); keys read 24 B and write
// 12 B per particle (on builds of up to about 4M particles the sort's first pass
// makes the keys as it loads the positions, see k_sort.hip). The AABB combines
// per-block partial extrema in a second one-block kernel (uses Device::diag, 6
// doubles per block, 1024 blocks).
#include "bh_internal.h"
#include "morton.h"

#include <cfloat>

namespace bh {
namespace {

__device__ inline double wave_min(double v)
{
    for (int o = 32; o > 0; o >>= 1)
        v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1)
        v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// Grid-stride min/max of the three FP64 coordinate arrays; each block writes
// its six partial extrema (no atomics; the final kernel combines them, so the
// result is deterministic).
__global__ __launch_bounds__(256) void aabb_kernel(const double* __restrict__ px,
                                                   const double* __restrict__ py,
                                                   const double* __restrict__ pz, size_t n,
                                                   double* __restrict__ partial)
{
    __shared__ double red[6][4];
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
    double hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += stride) {
        const double x = px[i], y = py[i], z = pz[i];
        lo[0] = fmin(lo[0], x);
        lo[1] = fmin(lo[1], y);
        lo[2] = fmin(lo[2], z);
        hi[0] = fmax(hi[0], x);
        hi[1] = fmax(hi[1], y);
        hi[2] = fmax(hi[2], z);
    }
    const int w = threadIdx.x >> 6;
    for (int a = 0; a < 3; ++a) {
        const double l = wave_min(lo[a]);
        const double h = wave_max(hi[a]);
        if ((threadIdx.x & 63) == 0) {
            red[a][w] = l;
            red[3 + a][w] = h;
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        double v = red[a][0];
        for (int k = 1; k < 4; ++k)
            v = a < 3 ? fmin(v, red[a][k]) : fmax(v, red[a][k]);
        partial[6 * blockIdx.x + a] = v;
    }
}

// Combine the per-block extrema and derive the root geometry (one block; the
// two took a launch each, about 4 us of a small build).
__global__ __launch_bounds__(256) void geometry_kernel(const double* __restrict__ partial, int nb,
                                                       RootGeom* __restrict__ g)
{
    __shared__ double red[6][4];
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
    double hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (int b = threadIdx.x; b < nb; b += blockDim.x)
        for (int a = 0; a < 3; ++a) {
            lo[a] = fmin(lo[a], partial[6 * b + a]);
            hi[a] = fmax(hi[a], partial[6 * b + 3 + a]);
        }
    const int w = threadIdx.x >> 6;
    for (int a = 0; a < 3; ++a) {
        const double l = wave_min(lo[a]);
        const double h = wave_max(hi[a]);
        if ((threadIdx.x & 63) == 0) {
            red[a][w] = l;
            red[3 + a][w] = h;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int a = threadIdx.x;
        double l = red[a][0], h = red[3 + a][0];
        for (int k = 1; k < 4; ++k) {
            l = fmin(l, red[a][k]);
            h = fmax(h, red[3 + a][k]);
        }
        const float flo = static_cast<float>(l);
        const float fhi = static_cast<float>(h);
        const float inv = __fdiv_rn(1.0f, fmaxf(fhi - flo, 1.0e-12f));
        g->lo[a] = flo;
        g->inv[a] = inv;
        // The lattice unit is half of one quantisation step of the FP32 frame:
        // step = 1 / (inv * (2^21 - 1)).
        const double step = 1.0 / (static_cast<double>(inv) * static_cast<double>(kQMax));
        g->lo_d[a] = static_cast<double>(flo);
        g->unit_d[a] = 0.5 * step;
        g->unit_f[a] = static_cast<float>(0.5 * step);
        g->width_f[a] = static_cast<float>(step);
    }
}

template <int MODE>
__global__ __launch_bounds__(256) void keys_kernel(const double* __restrict__ px,
                                                   const double* __restrict__ py,
                                                   const double* __restrict__ pz, size_t n,
                                                   const RootGeom* __restrict__ g,
                                                   unsigned long long* __restrict__ keys,
                                                   uint32_t* __restrict__ vals)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    keys[i] = morton_key<MODE>(px[i], py[i], pz[i], g);
    vals[i] = static_cast<uint32_t>(i);
}

}  // namespace

void launch_aabb(Device& d)
{
    int nb = d.aabb_parts;  // partials the drift kernel left for these positions
    d.aabb_parts = 0;
    if (nb <= 0) {
        const size_t blocks = std::min<size_t>((d.n + 255) / 256, kAabbBlocks);
        nb = static_cast<int>(std::max<size_t>(blocks, 1));
        aabb_kernel<<<nb, 256, 0, d.stream>>>(d.pos[0], d.pos[1], d.pos[2], d.n, d.diag);
    }
    geometry_kernel<<<1, 256, 0, d.stream>>>(d.diag, nb, d.geom);
}

void launch_keys(Device& d, int key_mode)
{
    const unsigned blocks = static_cast<unsigned>((d.n + 255) / 256);
    if (blocks == 0)
        return;
    if (key_mode == 1)
        keys_kernel<1><<<blocks, 256, 0, d.stream>>>(
            d.pos[0], d.pos[1], d.pos[2], d.n, d.geom,
            reinterpret_cast<unsigned long long*>(d.keys), d.vals);
    else
        keys_kernel<0><<<blocks, 256, 0, d.stream>>>(
            d.pos[0], d.pos[1], d.pos[2], d.n, d.geom,
            reinterpret_cast<unsigned long long*>(d.keys), d.vals);
}

}  // namespace bh
