// Wavefront-grouped Barnes-Hut walk for octree_hip.
//
// Reference semantics (per target, engine/physics/octree/traversal/
// OctreeTraversal.cpp:129-222 and engine/physics/octree/cuda/force/
// OctGpu.inl:100-228): skip empty nodes; a node is accepted as a single source
// at its centre of mass when the target is not inside it and
//   size / sqrt(|com - x|^2 + eps^2) < theta      (criterion "com"), or
//   size / dist(x, box)               < theta      (criterion "bounds");
// octree_hip adds criterion "extent": bmax / sqrt(|com - x|^2 + eps^2) < theta,
// bmax the radius about the COM that encloses the node's particles (the
// multipole truncation error scales with bmax / distance, not cell size);
// otherwise it is opened; particles of opened leaves are summed directly
// (pair force engine/physics/octree/force/OctreeForce.cpp:23-57); the sum is
// clamped to max_acceleration (engine/physics/octree/force/OctForces.cpp:128-133).
//
// MI355X mapping. One workgroup owns a group of at most 64 targets (one target
// per lane) -- the particles of one tree node, so the group is spatially compact
// -- and walks the tree once for the whole group: one wavefront where there are
// groups enough to fill the chip, 2, 4 or 8 that share the lists and the stack
// where there are not (walk_waves). A node is accepted only when the criterion holds for every
// point of the group's bounding box (distance measured from the box, which is
// conservative), and only when no target lies within the node's bounding
// sphere (bmax) -- the group form of the reference's "contains self" test.
// Accepted nodes (monopole + traceless quadrupole) and the particles of opened
// leaves are staged in LDS lists and evaluated by all lanes with broadcast LDS
// reads. Traversal keeps a LIFO of node indices, popped 64 per wavefront at a
// time, in global memory (its top in LDS where several wavefronts share it).
// Groups are handed out by an atomic ticket; every workgroup
// exits when the ticket passes the group count.
//
// Precision: positions in the walk are FP32 offsets from the exact lattice
// centre of the group's node: float(c_node - c_ref) * unit + offset,
// with integer lattice coordinates c, so the walk itself uses no FP64.
//
// Second order (multipole_order 2) is the expansion of the Plummer-softened
// kernel g(r) = (r^2 + eps^2)^-1/2 about the COM, d = com - x, R^2 = |d|^2 + eps^2:
//   a = M d / R^3 - Q d / R^5 + 5/2 (d.Q d - eps^2 trs) d / R^7,
// Q the traceless quadrupole, trs = sum m |y|^2 (the eps^2 trs term is what
// the traceless Q cannot carry once eps > 0). multipole_order 1 is the
// reference's softened monopole.
//
// Cost model for the roofline: 20 FLOP per particle-particle and 50 FLOP per
// particle-cell (monopole + quadrupole) interaction.
#include "bh_internal.h"

namespace bh {
namespace {

// LDS list capacities (cells flush at kCellCap - 64, particles at kPartCap);
// together with the leaf descriptors they set the LDS per wavefront and so
// the walk's residency: 96 and 96, cells of 48 bytes, take 7.4 KB (22 waves per
// CU by LDS, 20 by VGPRs in the relative walk). Chosen with cells of 40 bytes: 6.5 KB
// against 8.3 KB (18 waves per CU) for 128 and 128, the relative walk 2 % faster at 8M.
#ifndef BH_WALK_CELL_CAP
#define BH_WALK_CELL_CAP 96
#endif
#ifndef BH_WALK_PART_CAP
#define BH_WALK_PART_CAP 96
#endif
// Walks of W waves per group append up to 64 W entries per step, so their
// lists grow with W.
template <int W>
struct WalkCaps {
    static constexpr int kCell = W == 1 ? BH_WALK_CELL_CAP : 64 * W + 64;
    static constexpr int kPart = W == 1 ? BH_WALK_PART_CAP : 64 * W + 64;
    // stack entries below this depth live in LDS (W > 1)
    static constexpr int kLdsStack = W == 1 ? 0 : 256 * W;
};

// Group tickets. On large walks (at least kQueueMinGroupsPerWave groups per
// resident wave) the walk order is cut into chunks of kTicketChunk
// consecutive groups, dealt round-robin to kQueues counters; a wave draws
// from the queue of its XCD, so the groups one XCD walks at a time are
// neighbours in space and share tree nodes in that XCD's L2. Smaller walks
// use one counter: with few groups per wave, the per-XCD split costs more in
// balance than it gains in locality.
#ifndef BH_WALK_TICKET_QUEUES
#define BH_WALK_TICKET_QUEUES 8
#endif
#ifndef BH_WALK_TICKET_CHUNK
#define BH_WALK_TICKET_CHUNK 16
#endif
constexpr int kQueues = BH_WALK_TICKET_QUEUES;
constexpr unsigned kTicketChunk = BH_WALK_TICKET_CHUNK;
constexpr int kQueueMinGroupsPerWave = 16;
static_assert(kQueues >= 1 && kQueues <= kTicketQueues, "ticket queues");

// position in the walk order of the k-th ticket of queue q (of nq)
__device__ inline int ticket_position(unsigned k, int q, int nq)
{
    return static_cast<int>(((k / kTicketChunk) * static_cast<unsigned>(nq) +
                             static_cast<unsigned>(q)) * kTicketChunk + k % kTicketChunk);
}

// Group-box reductions, once per group. (Written with DPP row rotations and
// row broadcasts, each step waits on the one before; with the shuffles below
// other waves fill those waits, and the 1M-particle COM walk was 3 % faster.)
__device__ inline float wmin(float v)
{
    for (int o = 32; o > 0; o >>= 1)
        v = fminf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline float wmax(float v)
{
    for (int o = 32; o > 0; o >>= 1)
        v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
// Inclusive scan over the 64 lanes (all active) in six DPP adds: shifts of
// 1, 2, 4 and 8 within each 16-lane row, then lane 15 of each row into the
// next (rows 1 and 3) and lane 31 into rows 2 and 3. Lanes a shift leaves
// without a source, and rows the row mask excludes, add the old value 0.
// (Written with lane shuffles, each step is an LDS permute and a wait.)
__device__ inline uint32_t winclusive(uint32_t v)
{
    int x = static_cast<int>(v);
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return static_cast<uint32_t>(x);
}

// the value of lane 63 (a wave-uniform scalar)
__device__ inline uint32_t wlast(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// TreePM short-range weight of the Newtonian pair force:
// w(r) = erfc(r / 2rs) + r / (rs sqrt(pi)) exp(-r^2 / 4rs^2)
// (engine/physics/octree/force/OctreeForce.cpp:49-57). With x = r / rs it is
// E(x) Q(x), E = exp(-x^2 / 4) and Q(x) = erfcx(x / 2) + x / sqrt(pi) smooth
// (erfcx the scaled complementary error function). Q is this build's
// degree-13 least-squares polynomial on [0, 8] (Chebyshev points, weight E),
// held at x = 8 beyond: the FP32 evaluation errs by at most 1.6e-7 in w for
// every x (checked against erfc on the host). One exp2 and 13 FMAs against
// about 50 instructions for erfcf and expf.
__constant__ float kTpmQ[14] = {
    1.000000000e+00f,  2.537409785e-07f, 2.499964684e-01f,  -9.401225299e-02f,
    3.119471297e-02f,  -9.308321401e-03f, 2.498052781e-03f, -5.898143281e-04f,
    1.174437930e-04f,  -1.865963713e-05f, 2.218408781e-06f, -1.821118900e-07f,
    9.095778353e-09f,  -2.065529969e-10f};

// w(x) and E(x) = exp(-x^2 / 4), x = r / rs. The exponent comes from r^2 (r2, with
// e2 = -log2(e) / 4 rs^2) instead of x: one product less and one rounding less (w
// errs by at most 1.6e-7 instead of 2.2e-7, r and x rounded to FP32 included).
__device__ inline float tpm_weight_e(float x, float r2, float e2, float& E)
{
    const float xc = fminf(x, 8.0f);
    float q = kTpmQ[13];
#pragma unroll
    for (int k = 12; k >= 0; --k)
        q = fmaf(q, xc, kTpmQ[k]);
    E = __builtin_amdgcn_exp2f(r2 * e2);
    return q * E;
}

__device__ inline float tpm_e2(float inv_rs) { return -0.3606737554f * (inv_rs * inv_rs); }

// An accepted node in the cell list: (COM, mass), (qxx, qxy, qxz, qyy),
// (qyz, trs term, qzz, -). The trs term is eps^2 trs in the open walk, trs in the
// TreePM one.
struct Cell {
    float4 a, b, c;
};

// List evaluation. A lane takes entries j0, j0 + DJ, ...: one share of the list
// for groups of more than 32 targets walked by one wave; smaller groups give each
// target 2 or 4 lanes and W waves split each of those W ways (see walk_kernel); the
// shares are summed at the end of the group. The open walk's lists are padded with
// massless entries far away (pad_cells, pad_parts) to whole turns of DJ, and one
// share (DJ = 1) starts at entry 0: every lane makes the same number of turns, and
// the loop is counted in scalar registers. Counted per lane it took 2.2 VALU
// instructions of 36 per cell and 0.75 of 13.75 per particle.
constexpr uint32_t kHalfBox = 1u << 31;  // beside a wave's count of accepted cells
constexpr float kPadFar = 1.0e18f;  // its square is finite in FP32, its force zero

// WRAP: pairs take their nearest image (a periodic TreePM box). The walk shifts every
// node to the image nearest to the group, so a pair needs its own only where an entry
// lies half a box from some target (far_image in walk_kernel); elsewhere rounding the
// separation to whole boxes gives 0, and the loops without it sum the same terms (9 of
// 45 VALU instructions a particle less). With the shorter cells below: VALU instructions
// per 128^3 walk 1.77e9 -> 1.37e9, 2.42 -> 2.02 ms, still bound by VALU issue.
template <int ORDER, bool TPM, bool WRAP, int DJ>
__device__ inline void eval_cells_dj(const Cell* __restrict__ cl, int ncell, int j0, float tx,
                                     float ty, float tz, const WalkParams& P, float& ax, float& ay,
                                     float& az)
{
    // (a compile-time stride keeps the unrolled LDS reads on one base)
    const int turns = DJ == 1 || !TPM ? (ncell + DJ - 1) / DJ : (ncell - j0 + DJ - 1) / DJ;
    const Cell* p = DJ == 1 ? cl : cl + j0;
    const float inv_rs = TPM ? 1.0f / P.rs : 0.0f;
    const float e2 = TPM ? tpm_e2(inv_rs) : 0.0f;
    const float cE = 0.28209479177387814f * inv_rs * inv_rs * inv_rs;  // 1 / (2 sqrt(pi) rs^3)
    const float cE2 = 0.25f * inv_rs * inv_rs * cE;
    const float box = WRAP ? P.box : 0.0f;
    const float ib = WRAP ? 1.0f / box : 0.0f;
#pragma unroll 2
    for (int k = 0; k < turns; ++k, p += DJ) {
        const float4 a = p->a;
        float dx = a.x - tx, dy = a.y - ty, dz = a.z - tz;
        if (WRAP) {  // nearest image of this pair
            dx -= box * rintf(dx * ib);
            dy -= box * rintf(dy * ib);
            dz -= box * rintf(dz * ib);
        }
        const float r2 = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, P.eps2)));
        const float ri = __frsqrt_rn(r2);
        const float ri2 = ri * ri;
        const float ri3 = ri * ri2;
        float wgt = 1.0f, E;
        if (TPM && ORDER < 2)
            wgt = tpm_weight_e(r2 * ri * inv_rs, r2, e2, E);
        if (TPM && ORDER >= 2) {
            // Second-order expansion of the short-range kernel g(R) d,
            // g = w(R) / R^3, about the COM (S = (Q + trs I) / 3 the raw
            // second moment, Q traceless):
            //   a = [M g + G2 (dQd + trs |d|^2) / 6 + 5/6 G1 trs] d + G1 / 3 Q d
            // with G1 = g'(R) / R, G2 = G1'(R) / R. For the erfc weight,
            // w'(R) = -R^2 E / (2 sqrt(pi) rs^3), E = exp(-R^2 / 4 rs^2), so
            // with c = E / (2 sqrt(pi) rs^3)
            //   u = -G1 = (c + 3 g) / R^2,
            //   G2 = (c / (2 rs^2) + 5 u) / R^2.
            // With w = 1, c = 0 it is the softened Newtonian expansion of the open
            // walk. The list holds Q / 3, trs / 3 and 5/6 trs, so that no factor is
            // left over: 56 VALU instructions a cell against 66.
            const float4 b = p->b;
            const float4 c = p->c;  // (qyz, trs, qzz) / 3, 5/6 trs
            const float qx = fmaf(b.z, dz, fmaf(b.y, dy, b.x * dx));
            const float qy = fmaf(c.x, dz, fmaf(b.w, dy, b.y * dx));
            const float qz = fmaf(c.z, dz, fmaf(c.x, dy, b.z * dx));
            const float w = tpm_weight_e(r2 * ri * inv_rs, r2, e2, E);
            const float g = w * ri3;
            const float u = fmaf(3.0f, g, E * cE) * ri2;
            const float h = fmaf(2.5f, u, E * cE2) * ri2;  // G2 / 2
            const float d2 = r2 - P.eps2;
            const float q2 = fmaf(dz, qz, fmaf(dy, qy, fmaf(dx, qx, c.y * d2)));
            const float s = fmaf(h, q2, fmaf(a.w, g, -(c.w * u)));
            ax = fmaf(-u, qx, fmaf(s, dx, ax));
            ay = fmaf(-u, qy, fmaf(s, dy, ay));
            az = fmaf(-u, qz, fmaf(s, dz, az));
        } else if (ORDER >= 2) {
            const float4 b = p->b;
            const float4 c = p->c;
            // b = (qxx, qxy, qxz, qyy), c = (qyz, eps^2 trs, qzz)
            const float qx = fmaf(b.z, dz, fmaf(b.y, dy, b.x * dx));
            const float qy = fmaf(c.x, dz, fmaf(b.w, dy, b.y * dx));
            const float qz = fmaf(c.z, dz, fmaf(c.x, dy, b.z * dx));
            const float dqd = fmaf(dz, qz, fmaf(dy, qy, dx * qx));
            // M/R^3 + 5/2 (dQd - eps^2 trs)/R^7 = (M + 5/2 (dQd - eps^2 trs)/R^4) / R^3
            const float u = (dqd - c.y) * ri2;
            const float s = fmaf(2.5f * u, ri2, a.w) * ri3 * wgt;
            const float t = ri3 * ri2 * wgt;
            ax = fmaf(-t, qx, fmaf(s, dx, ax));
            ay = fmaf(-t, qy, fmaf(s, dy, ay));
            az = fmaf(-t, qz, fmaf(s, dz, az));
        } else {
            const float s = a.w * ri3 * wgt;
            ax += s * dx;
            ay += s * dy;
            az += s * dz;
        }
    }
}

template <bool TPM, bool WRAP, int DJ>
__device__ inline void eval_parts_dj(const float4* __restrict__ pl, int np, int j0, float tx,
                                     float ty, float tz, const WalkParams& P, float& ax, float& ay,
                                     float& az)
{
    const int turns = DJ == 1 || !TPM ? (np + DJ - 1) / DJ : (np - j0 + DJ - 1) / DJ;
    const float4* p = DJ == 1 ? pl : pl + j0;
    if (!TPM && P.eps2 > 0.0f && P.min_d2 <= P.eps2) {
        // every pair has r2 >= eps2 >= min_d2: the skip test can only drop a
        // coincident pair, whose contribution is exactly zero anyway
        const float eps2 = P.eps2;
#pragma unroll 4
        for (int k = 0; k < turns; ++k, p += DJ) {
            const float4 a = *p;
            const float dx = a.x - tx, dy = a.y - ty, dz = a.z - tz;
            const float r2 = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, eps2)));
            const float ri = __frsqrt_rn(r2);
            const float s = a.w * ri * (ri * ri);
            ax += s * dx;
            ay += s * dy;
            az += s * dz;
        }
        return;
    }
    const float inv_rs = TPM ? 1.0f / P.rs : 0.0f;
    const float e2 = TPM ? tpm_e2(inv_rs) : 0.0f;
    const float box = WRAP ? P.box : 0.0f;
    const float ib = WRAP ? 1.0f / box : 0.0f;
    const float cut2 = TPM && P.rcut2 > 0.0f ? P.rcut2 : __builtin_inff();
#pragma unroll 4
    for (int k = 0; k < turns; ++k, p += DJ) {
        const float4 a = *p;
        float dx = a.x - tx, dy = a.y - ty, dz = a.z - tz;
        if (WRAP) {  // nearest image of this pair
            dx -= box * rintf(dx * ib);
            dy -= box * rintf(dy * ib);
            dz -= box * rintf(dz * ib);
        }
        // (the order of the sum is that of every loop here: a pair at the cutoff is
        // in or out by its last bit)
        const float d2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        const float r2 = d2 + P.eps2;
        const float ri = __frsqrt_rn(r2);
        // (both tests without a branch: a wavefront hardly ever drops all of a pair)
        const bool use = (r2 > P.min_d2) & (!TPM || d2 <= cut2);
        float s = a.w * ri * ri * ri;
        if (TPM) {
            float E;
            s *= tpm_weight_e(r2 * ri * inv_rs, r2, e2, E);
        }
        s = use ? s : 0.0f;
        ax += s * dx;
        ay += s * dy;
        az += s * dz;
    }
}

// Whole turns of dj * W entries: massless ones after the last (the capacities
// are multiples of 4 W). A barrier follows where there are several shares.
template <bool TPM, int W>
__device__ inline void pad_cells(Cell* cl, int n, int dj)
{
    if (TPM || W * dj == 1)
        return;
    const int at = n + static_cast<int>(threadIdx.x);
    if (at < (n + dj * W - 1) / (dj * W) * (dj * W)) {
        cl[at].a = make_float4(kPadFar, kPadFar, kPadFar, 0.0f);
        cl[at].b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        cl[at].c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    __syncthreads();
}
template <bool TPM, int W>
__device__ inline void pad_parts(float4* pl, int n, int dj)
{
    if (TPM || W * dj == 1)
        return;
    const int at = n + static_cast<int>(threadIdx.x);
    if (at < (n + dj * W - 1) / (dj * W) * (dj * W))
        pl[at] = make_float4(kPadFar, kPadFar, kPadFar, 0.0f);
    __syncthreads();
}

template <int ORDER, bool TPM, bool WRAP, int W>
__device__ inline void eval_cells_w(const Cell* __restrict__ cl, int ncell, int j0, int dj,
                                    float tx, float ty, float tz, const WalkParams& P, float& ax,
                                    float& ay, float& az)
{
    if (dj == 1)
        eval_cells_dj<ORDER, TPM, WRAP, W>(cl, ncell, j0, tx, ty, tz, P, ax, ay, az);
    else if (dj == 2)
        eval_cells_dj<ORDER, TPM, WRAP, 2 * W>(cl, ncell, j0, tx, ty, tz, P, ax, ay, az);
    else
        eval_cells_dj<ORDER, TPM, WRAP, 4 * W>(cl, ncell, j0, tx, ty, tz, P, ax, ay, az);
}

template <int ORDER, bool TPM, int W>
__device__ inline void eval_cells(Cell* __restrict__ cl, int ncell, int j0, int dj, bool wrap,
                                  float tx, float ty, float tz, const WalkParams& P, float& ax,
                                  float& ay, float& az)
{
    pad_cells<TPM, W>(cl, ncell, dj);
    if (TPM && wrap)
        eval_cells_w<ORDER, TPM, TPM, W>(cl, ncell, j0, dj, tx, ty, tz, P, ax, ay, az);
    else
        eval_cells_w<ORDER, TPM, false, W>(cl, ncell, j0, dj, tx, ty, tz, P, ax, ay, az);
}

template <bool TPM, bool WRAP, int W>
__device__ inline void eval_parts_w(const float4* __restrict__ pl, int np, int j0, int dj,
                                    float tx, float ty, float tz, const WalkParams& P, float& ax,
                                    float& ay, float& az)
{
    if (dj == 1)
        eval_parts_dj<TPM, WRAP, W>(pl, np, j0, tx, ty, tz, P, ax, ay, az);
    else if (dj == 2)
        eval_parts_dj<TPM, WRAP, 2 * W>(pl, np, j0, tx, ty, tz, P, ax, ay, az);
    else
        eval_parts_dj<TPM, WRAP, 4 * W>(pl, np, j0, tx, ty, tz, P, ax, ay, az);
}

template <bool TPM, int W>
__device__ inline void eval_parts(float4* __restrict__ pl, int np, int j0, int dj, bool wrap,
                                  float tx, float ty, float tz, const WalkParams& P, float& ax,
                                  float& ay, float& az)
{
    pad_parts<TPM, W>(pl, np, dj);
    if (TPM && wrap)
        eval_parts_w<TPM, TPM, W>(pl, np, j0, dj, tx, ty, tz, P, ax, ay, az);
    else
        eval_parts_w<TPM, false, W>(pl, np, j0, dj, tx, ty, tz, P, ax, ay, az);
}

// Group far field: the local (Taylor) expansion about the group centre of an
// accepted node's softened second-order field,
//   a(g + delta) = A + J delta + 1/2 H delta delta,
// r = COM - g, R^2 = |r|^2 + eps^2, S = (Q + trs I)/3:
//   A_i  = M r_i R^-3 + 7.5 (rSr) r_i R^-7 - 3 (Sr)_i R^-5 - 1.5 trs r_i R^-5
//   J_il = M (3 r_i r_l R^-5 - d_il R^-3)
//          + (52.5 rSr R^-9 - 7.5 trs R^-7) r_i r_l - 15 R^-7 ((Sr)_i r_l + (Sr)_l r_i)
//          + d_il (1.5 trs R^-5 - 7.5 rSr R^-7) + 3 R^-5 S_il
//   H_ijk = M (15 r_i r_j r_k R^-7 - 3 (d_ij r_k + d_ik r_j + d_jk r_i) R^-5)
// (the monopole to second order in delta, the quadrupole to first).
// Storage: F[0..2] A, F[3..8] J (xx xy xz yy yz zz), F[9..18] H (xxx xxy xxz xyy
// xyz xzz yyy yyz yzz zzz).
constexpr int kFarTerms = 19;
#ifndef BH_FAR_GROUP_WEIGHT
#define BH_FAR_GROUP_WEIGHT 3.0f
#endif
constexpr float kFarGroupWeight = BH_FAR_GROUP_WEIGHT;

__device__ inline void far_accumulate(float rx, float ry, float rz, const WalkNode& w, float eps2,
                                      float* F)
{
    const float R2 = rx * rx + ry * ry + rz * rz + eps2;
    const float ri = __frsqrt_rn(R2);
    const float ri2 = ri * ri;
    const float ri3 = ri * ri2, ri5 = ri3 * ri2, ri7 = ri5 * ri2, ri9 = ri7 * ri2;
    const float M = w.mass, t = w.trs;
    const float third = 1.0f / 3.0f;
    const float sxx = (w.qxx + t) * third, syy = (w.qyy + t) * third;
    const float szz = (-w.qxx - w.qyy + t) * third;
    const float sxy = w.qxy * third, sxz = w.qxz * third, syz = w.qyz * third;
    const float qx = sxx * rx + sxy * ry + sxz * rz;
    const float qy = sxy * rx + syy * ry + syz * rz;
    const float qz = sxz * rx + syz * ry + szz * rz;
    const float rsr = rx * qx + ry * qy + rz * qz;
    // A
    const float am = M * ri3 + 7.5f * rsr * ri7 - 1.5f * t * ri5;
    F[0] += am * rx - 3.0f * ri5 * qx;
    F[1] += am * ry - 3.0f * ri5 * qy;
    F[2] += am * rz - 3.0f * ri5 * qz;
    // J
    const float jr = 3.0f * M * ri5 + 52.5f * rsr * ri9 - 7.5f * t * ri7;
    const float jd = -M * ri3 + 1.5f * t * ri5 - 7.5f * rsr * ri7;
    const float js = 3.0f * ri5, jq = -15.0f * ri7;
    F[3] += jr * rx * rx + jq * 2.0f * qx * rx + jd + js * sxx;
    F[4] += jr * rx * ry + jq * (qx * ry + qy * rx) + js * sxy;
    F[5] += jr * rx * rz + jq * (qx * rz + qz * rx) + js * sxz;
    F[6] += jr * ry * ry + jq * 2.0f * qy * ry + jd + js * syy;
    F[7] += jr * ry * rz + jq * (qy * rz + qz * ry) + js * syz;
    F[8] += jr * rz * rz + jq * 2.0f * qz * rz + jd + js * szz;
    // H
    const float c7 = 15.0f * M * ri7, c5 = 3.0f * M * ri5;
    F[9] += (c7 * rx * rx - 3.0f * c5) * rx;
    F[10] += (c7 * rx * rx - c5) * ry;
    F[11] += (c7 * rx * rx - c5) * rz;
    F[12] += (c7 * ry * ry - c5) * rx;
    F[13] += c7 * rx * ry * rz;
    F[14] += (c7 * rz * rz - c5) * rx;
    F[15] += (c7 * ry * ry - 3.0f * c5) * ry;
    F[16] += (c7 * ry * ry - c5) * rz;
    F[17] += (c7 * rz * rz - c5) * ry;
    F[18] += (c7 * rz * rz - 3.0f * c5) * rz;
}

__device__ inline void far_evaluate(const float* F, float dx, float dy, float dz, float& ax,
                                    float& ay, float& az)
{
    const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
    const float xy = dx * dy, xz = dx * dz, yz = dy * dz;
    ax += F[0] + F[3] * dx + F[4] * dy + F[5] * dz +
          0.5f * (F[9] * xx + F[12] * yy + F[14] * zz) + F[10] * xy + F[11] * xz + F[13] * yz;
    ay += F[1] + F[4] * dx + F[6] * dy + F[7] * dz +
          0.5f * (F[10] * xx + F[15] * yy + F[17] * zz) + F[12] * xy + F[13] * xz + F[16] * yz;
    az += F[2] + F[5] * dx + F[7] * dy + F[8] * dz +
          0.5f * (F[11] * xx + F[16] * yy + F[18] * zz) + F[13] * xy + F[14] * xz + F[17] * yz;
}

// Far nodes of a group are queued in LDS (node indices) and folded into the
// group's expansion in batches of up to kFarCap, with every lane taking whole
// nodes; the lanes' partial sums are reduced once per batch into fsum. The
// 19 accumulators are then live only inside the batch, not across the list
// evaluation loops.
constexpr int kFarCap = 256;

__device__ inline void far_flush(const uint32_t* __restrict__ fl, int nfl,
                                 const WalkNode* __restrict__ nodes, int rcx, int rcy, int rcz,
                                 float ux, float uy, float uz, float gcx, float gcy, float gcz,
                                 float eps2, float* __restrict__ fsum)
{
    float F[kFarTerms];
#pragma unroll
    for (int k = 0; k < kFarTerms; ++k)
        F[k] = 0.0f;
#pragma unroll 1
    for (int i = static_cast<int>(threadIdx.x); i < nfl; i += 64) {
        const WalkNode w = nodes[fl[i]];
        const float rx = static_cast<float>(w.cx - rcx) * ux + w.comx - gcx;
        const float ry = static_cast<float>(w.cy - rcy) * uy + w.comy - gcy;
        const float rz = static_cast<float>(w.cz - rcz) * uz + w.comz - gcz;
        far_accumulate(rx, ry, rz, w, eps2, F);
    }
#pragma unroll
    for (int k = 0; k < kFarTerms; ++k) {
        float v = F[k];
        for (int o = 32; o > 0; o >>= 1)
            v += __shfl_xor(v, o, 64);
        F[k] = v;
    }
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < kFarTerms; ++k)
            fsum[k] += F[k];
    }
}

// Pushes nodes first, first + 1, ... (1 to 8 of them) by at most three stores. One store
// per child took as many turns as the wavefront's largest nc, of 6 VALU instructions.
// With the leaf search below 44 of about 190 VALU instructions per traversal step: a
// 65,536-particle step 624 -> 613 us, 128^3 TreePM forces 3.62 -> 3.52 ms.
__device__ inline void push_children(int* __restrict__ to, int first, uint32_t nc)
{
    typedef int int4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef int int2_a4 __attribute__((ext_vector_type(2), aligned(4)));
    if (nc >= 4u) {
        *reinterpret_cast<int4_a4*>(to) = int4_a4{first, first + 1, first + 2, first + 3};
        to += 4;
        first += 4;
        nc -= 4u;
    }
    if (nc == 4u) {
        *reinterpret_cast<int4_a4*>(to) = int4_a4{first, first + 1, first + 2, first + 3};
        return;
    }
    if (nc & 2u) {
        *reinterpret_cast<int2_a4*>(to) = int2_a4{first, first + 1};
        to += 2;
        first += 2;
    }
    if (nc & 1u)
        *to = first;
}

// W waves walk one group together (W > 1: small walks, see walk_waves). They
// pop up to 64 W nodes per step, share the lists in LDS, take every W-th
// entry of them each and add their shares of a target's force in wave order at
// the end, so results do not depend on timing. The nodes accepted and opened
// are those of the one-wave walk. Bound: latency (a step is one round trip for
// its nodes, one for the particles of opened leaves and 4 barriers, about 3.5 us
// for 256 nodes with 4 waves; about 10 steps per group at 4,096 particles).
// Issuing a step's node loads before the evaluation of the step before it
// changed nothing with 4 waves and cost 10 % with 2.
template <int ORDER, int CRIT, bool TPM, bool REC, bool FAR, int W>
#ifndef BH_WALK_MIN_WAVES
#define BH_WALK_MIN_WAVES 5
#endif
// Walks without the far field are held to 96 VGPRs (5 waves per SIMD): the
// traversal is latency-bound and needs the resident waves.
__global__ __launch_bounds__(64 * W, FAR ? 1 : W > 1 ? 4 : BH_WALK_MIN_WAVES) void walk_kernel(
    WalkParams P, const WalkNode* __restrict__ nodes, const float4* __restrict__ spart,
    const uint32_t* __restrict__ sleaf, const RootGeom* __restrict__ geom,
    const uint4* __restrict__ groups, const int* __restrict__ info,
    int node_cap, unsigned int* __restrict__ work, int* __restrict__ stack_all, int stack_cap,
    float* __restrict__ accx, float* __restrict__ accy, float* __restrict__ accz,
    int* __restrict__ err, unsigned long long* __restrict__ stats, uint32_t* __restrict__ rec_lists,
    uint32_t* __restrict__ rec_n, int rec_cap, int rec_groups, float rec_band2,
    uint32_t rec_min_count)
{
    static_assert(W == 1 || !FAR, "the group far field walks with one wave");
    constexpr int kCellCap = WalkCaps<W>::kCell;
    constexpr int kPartCap = WalkCaps<W>::kPart;
    constexpr int kLdsStack = WalkCaps<W>::kLdsStack;
    constexpr int kThreads = 64 * W;
    __shared__ Cell cl[kCellCap];
    __shared__ float4 pl[kPartCap];
    __shared__ int lfFirst[kThreads];
    __shared__ uint32_t lfPre[kThreads];
    __shared__ float lfSx[kThreads], lfSy[kThreads], lfSz[kThreads];
    __shared__ int lstk[W > 1 ? kLdsStack : 1];
    __shared__ uint32_t wtot[W > 1 ? W : 1][6];  // per wave: totals of one step
    __shared__ int sticket;
    __shared__ uint32_t fl[FAR ? kFarCap : 1];
    __shared__ float fsum[FAR ? kFarTerms : 1];

    const int lane = threadIdx.x & 63;
    const int wv =
        W == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    // W waves share W stack regions
    stack_cap *= W;
    int* stk = stack_all + static_cast<size_t>(blockIdx.x) * static_cast<size_t>(stack_cap);
    const float ux = geom->unit_f[0], uy = geom->unit_f[1], uz = geom->unit_f[2];
    const float wfx = geom->width_f[0], wfy = geom->width_f[1], wfz = geom->width_f[2];
    const float wfmax = fmaxf(fmaxf(wfx, wfy), wfz);
    const float rcut = TPM && P.rcut2 > 0.0f ? sqrtf(P.rcut2) : 0.0f;
    const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    unsigned long long npp = 0, npc = 0;
    // this wave's interaction totals, added to `stats` once when it exits
    // (one set of atomics per wave instead of per group: the counters are
    // single addresses every wave would otherwise contend for)
    unsigned long long tot_pp = 0, tot_pc = 0, tot_mono = 0, tot_far = 0, tot_eval = 0;
    const int ngroups = info[kInfoGroups];

    // A wave draws from its XCD's queue and, once that is drained, from the
    // others in turn; every queue position below ngroups is handed out exactly
    // once. (A ticket is drawn only when the wave is free: a wave that held
    // its next group while walking the current one would keep that group from
    // an idle wave at the end of the walk.)
    const int nq = static_cast<long long>(ngroups) >=
                           static_cast<long long>(kQueueMinGroupsPerWave) * gridDim.x
                       ? kQueues
                       : 1;
    int queue = static_cast<int>(blockIdx.x % static_cast<unsigned>(nq));
    int drained = 0;
    for (;;) {
        int t = ngroups;
        if (threadIdx.x == 0) {
            for (;;) {
                t = ticket_position(atomicAdd(&work[queue * kTicketStride], 1u), queue, nq);
                if (t < ngroups || drained == nq - 1)
                    break;
                ++drained;
                queue = (queue + 1) % nq;
            }
            t = t < ngroups ? t : ngroups;
        }
        if (W > 1) {
            __syncthreads();  // every wave has read the ticket before
            if (threadIdx.x == 0)
                sticket = t;
            __syncthreads();
            t = sticket;
        }
        // the whole wave is active here, so the first lane is lane 0
        const int ticket = __builtin_amdgcn_readfirstlane(t);
        if (ticket >= ngroups)
            break;
        // Groups are stored in the breadth-first order of their nodes, shallow
        // (sparse, cheap) levels first; taking them deepest first puts the
        // expensive dense groups at the start instead of in the tail.
        const int g = ngroups - 1 - ticket;

        const uint4 gr = groups[g];
        int nact = static_cast<int>(gr.y);
        // Targets of this walk: the group's particles, or under block time
        // steps those due a force now. The box, the relative tolerance and
        // the stored forces cover these only (the corrector reads no other
        // particle's force, and each particle is due again before its next
        // kick), so a group with a few due particles walks with their box.
        // The due particles are compacted to the first lanes (their offsets
        // pass through lfFirst, unused until the traversal), so that a group
        // with few of them splits its lists like a small group.
        if (P.alevel) {
            bool due = false;
            if (lane < nact) {
                const uint32_t lv = min(P.alevel[gr.x + static_cast<uint32_t>(lane)],
                                        static_cast<uint32_t>(P.alevels));
                due = (P.atick & ((1u << (static_cast<uint32_t>(P.alevels) - lv)) - 1u)) == 0u;
            }
            const unsigned long long dm = __ballot(due);
            if (dm == 0ull)
                continue;
            if (due && wv == 0)
                lfFirst[__popcll(dm & lt)] = lane;
            nact = static_cast<int>(__popcll(dm));
            __syncthreads();
        }
        // groups of <= 32 (<= 16) targets: 2 (4) lanes per target, each
        // evaluating every 2nd (4th) list entry
        const int dj = nact <= 16 ? 4 : (nact <= 32 ? 2 : 1);
        const int tw = 64 / dj;  // lanes per list share
        const int tl = lane & (tw - 1);
        const int j0 = lane / tw + dj * wv;
        const bool active = tl < nact;
        const int s = static_cast<int>(gr.x) + (P.alevel ? (active ? lfFirst[tl] : 0) : tl);
        const bool target = active;
        const int gnode = static_cast<int>(gr.z);
        const int rcx = nodes[gnode].cx, rcy = nodes[gnode].cy, rcz = nodes[gnode].cz;

        float tx = 0.0f, ty = 0.0f, tz = 0.0f;
        if (active) {
            const float4 p = spart[s];
            const int lf = static_cast<int>(sleaf[s]);
            tx = rel_pos(nodes[lf].cx - rcx, ux, p.x);
            ty = rel_pos(nodes[lf].cy - rcy, uy, p.y);
            tz = rel_pos(nodes[lf].cz - rcz, uz, p.z);
        }
        const float gx0 = wmin(target ? tx : 3.0e38f), gx1 = wmax(target ? tx : -3.0e38f);
        const float gy0 = wmin(target ? ty : 3.0e38f), gy1 = wmax(target ? ty : -3.0e38f);
        const float gz0 = wmin(target ? tz : 3.0e38f), gz1 = wmax(target ? tz : -3.0e38f);
        const float gcx = 0.5f * (gx0 + gx1), gcy = 0.5f * (gy0 + gy1), gcz = 0.5f * (gz0 + gz1);
        const float ghx = 0.5f * (gx1 - gx0), ghy = 0.5f * (gy1 - gy0), ghz = 0.5f * (gz1 - gz0);
        // relative criterion: the group's smallest |a| of the last evaluation,
        // floored at 1 % of its largest (a target whose force nearly cancels
        // has no meaningful relative error and would open everything)
        float rtol = 0.0f, rtol_mono = 0.0f;
        if (CRIT == 3) {
            const float am = target ? P.amag[s] : 0.0f;
            const float amin = wmin(target ? am : 3.0e38f), amax = wmax(am);
            rtol = P.ralpha * fmaxf(amin, 0.01f * amax);
            rtol_mono = P.rmono * rtol;
        }
        unsigned long long nmono = 0;

        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        const float grad = FAR ? sqrtf(ghx * ghx + ghy * ghy + ghz * ghz) : 0.0f;
        unsigned long long nfar = 0;
        int nfl = 0;
        if (FAR && lane < kFarTerms)
            fsum[lane] = 0.0f;
        int ncell = 0, npart = 0;
        int nrec = 0;
        // TreePM: some entry lies half a box or more from some target (uniform)
        bool far_image = false;
        int sp = 1;
        if (threadIdx.x == 0) {
            if (W > 1)
                lstk[0] = 0;
            else
                stk[0] = 0;  // root
        }
        __syncthreads();

        // Every iteration pops at least one node and a node is pushed at most
        // once per group in a well-formed tree, so node_cap iterations bound
        // the loop; the guard also stops a malformed tree from spinning.
        int iters = 0;
        while (sp > 0) {
            if (++iters > node_cap) {
                if (threadIdx.x == 0)
                    atomicOr(err, kErrStackOverflow);
                break;
            }
            const int take = sp < kThreads ? sp : kThreads;
            sp -= take;
            int node = -1;
            if (static_cast<int>(threadIdx.x) < take) {
                const int at = sp + static_cast<int>(threadIdx.x);
                node = W > 1 && at < kLdsStack ? lstk[W > 1 ? at : 0] : stk[at];
            }
            if (node >= node_cap) {
                atomicOr(err, kErrStackOverflow);
                node = -1;
            }
            __syncthreads();

            bool accept = false, direct = false, open = false, mono = false;
            WalkNode w = {};
            float sx = 0.0f, sy = 0.0f, sz = 0.0f;
            float px = 0.0f, py = 0.0f, pz = 0.0f;
            float size = 0.0f;
            bool near = false;
            bool wide = false;
            if (node >= 0) {
                w = nodes[node];
                if (w.mass > 0.0f) {
                    sx = static_cast<float>(w.cx - rcx) * ux;
                    sy = static_cast<float>(w.cy - rcy) * uy;
                    sz = static_cast<float>(w.cz - rcz) * uz;
                    px = sx + w.comx;
                    py = sy + w.comy;
                    pz = sz + w.comz;
                    if (TPM && P.box > 0.0f) {
                        if (4.0f * w.bmax > P.box) {
                            wide = true;  // spans several images: always opened
                        } else {
                            // the node's image nearest to the group
                            const float ib = 1.0f / P.box;
                            const float hx = -P.box * rintf((px - gcx) * ib);
                            const float hy = -P.box * rintf((py - gcy) * ib);
                            const float hz = -P.box * rintf((pz - gcz) * ib);
                            sx += hx;
                            sy += hy;
                            sz += hz;
                            px += hx;
                            py += hy;
                            pz += hz;
                        }
                    }
                    const float dx = fmaxf(fabsf(px - gcx) - ghx, 0.0f);
                    const float dy = fmaxf(fabsf(py - gcy) - ghy, 0.0f);
                    const float dz = fmaxf(fabsf(pz - gcz) - ghz, 0.0f);
                    const float d2 = dx * dx + dy * dy + dz * dz;
                    bool ok = d2 > w.bmax * w.bmax;
                    const int lvl = static_cast<int>(meta_level(w.meta));
                    size = cell_size(wfmax, lvl);
                    if (CRIT == 1) {
                        const float hs = ldexpf(0.5f, kMaxLevel - lvl);
                        const float bx = fmaxf(fabsf(sx - gcx) - ghx - hs * wfx, 0.0f);
                        const float by = fmaxf(fabsf(sy - gcy) - ghy - hs * wfy, 0.0f);
                        const float bz = fmaxf(fabsf(sz - gcz) - ghz - hs * wfz, 0.0f);
                        const float b2 = bx * bx + by * by + bz * bz;
                        ok = ok && b2 > 0.0f && size * size < P.theta2 * b2;
                    } else if (CRIT == 2) {
                        ok = ok && w.bmax * w.bmax < P.theta2 * (d2 + P.eps2);
                    } else if (CRIT == 3) {
                        const float r2 = d2 + P.eps2;
                        const float b2 = w.bmax * w.bmax;
                        const float err = ORDER >= 2 ? w.mass * b2 * w.bmax : w.mass * b2;
                        // (v_sqrt_f32: the acceptance needs no correctly rounded root)
                        const float lim = ORDER >= 2 ? rtol * r2 * r2 * __builtin_amdgcn_sqrtf(r2)
                                                     : rtol * r2 * r2;
                        ok = ok && size * size < P.theta2 * r2 && err <= lim;
                        // quadrupole term within tolerance too: a point mass suffices
                        mono = ORDER >= 2 && ok && w.mass * b2 <= rtol_mono * r2 * r2;
                    } else {
                        ok = ok && size * size < P.theta2 * (d2 + P.eps2);
                    }
                    if (TPM && P.rcut2 > 0.0f && !wide) {
                        // Prune nodes whose bounding sphere lies beyond the cutoff for the
                        // whole group.
                        const float lim = rcut + w.bmax;
                        if (d2 > lim * lim) {
                            ok = false;
                            w.mass = 0.0f;
                        }
                    }
                    if (wide)
                        ok = false;
                    if (REC && ok) {
                        // near the group: small nodes are opened, large ones
                        // accepted and recorded for the learned correction
                        // (a group beyond the lists' capacity opens them all)
                        near = size * size >= rec_band2 * d2;
                        if (near && (meta_count(w.meta) < rec_min_count || g >= rec_groups)) {
                            ok = false;
                            near = false;
                        }
                    }
                    if (w.mass > 0.0f) {
                        const uint32_t nch = meta_nchild(w.meta);
                        accept = ok;
                        direct = !ok && nch == 0;
                        open = !ok && nch != 0;
                    }
                }
            }
            bool half_box = false;  // of what this wave adds
            if (TPM && P.box > 0.0f) {
                const float reach = fmaxf(fmaxf(fabsf(px - gcx) + ghx, fabsf(py - gcy) + ghy),
                                          fabsf(pz - gcz) + ghz) + w.bmax;
                half_box = __ballot((accept || direct) && reach >= 0.49f * P.box) != 0ull;
                if (W == 1)
                    far_image = far_image || half_box;
            }

            if (REC) {
                near = near && accept;
                const unsigned long long rm = __ballot(near);
                int nnear = static_cast<int>(__popcll(rm));
                int before = 0;  // near nodes of the waves before this one
                if (W > 1) {
                    if (lane == 0)
                        wtot[wv][5] = static_cast<uint32_t>(nnear);
                    __syncthreads();
                    nnear = 0;
#pragma unroll
                    for (int k = 0; k < W; ++k) {
                        before += k < wv ? static_cast<int>(wtot[k][5]) : 0;
                        nnear += static_cast<int>(wtot[k][5]);
                    }
                }
                if (near) {
                    const int slot = nrec + before + static_cast<int>(__popcll(rm & lt));
                    if (slot < rec_cap) {
                        rec_lists[static_cast<size_t>(g) * rec_cap + slot] =
                            static_cast<uint32_t>(node);
                    } else {
                        // the group's list is full: open the node instead
                        // (its error is then the plain walk's, never an
                        // uncorrected near node's)
                        const uint32_t nch = meta_nchild(w.meta);
                        accept = false;
                        direct = nch == 0;
                        open = nch != 0;
                    }
                }
                nrec += nnear;
            }

            if (FAR) {
                // far from the whole group: queued for the group's local
                // expansion instead of the per-target list. The group radius
                // weighs kFarGroupWeight times the node's: the expansion is
                // second order in the offset from the group centre, with a
                // larger error constant than the node's own second-order
                // multipole.
                bool far = false;
                if (accept) {
                    const float rx = px - gcx, ry = py - gcy, rz = pz - gcz;
                    const float lim = w.bmax + kFarGroupWeight * grad;
                    far = lim * lim < P.far2 * (rx * rx + ry * ry + rz * rz);
                    accept = accept && !far;
                }
                const unsigned long long fm = __ballot(far);
                if (far)
                    fl[nfl + static_cast<int>(__popcll(fm & lt))] = static_cast<uint32_t>(node);
                nfl += static_cast<int>(__popcll(fm));
                nfar += __popcll(fm);
            }

            // What this step adds: counts per wave, then (W > 1) the offsets of
            // the waves before.
            if (CRIT == 3) {
                mono = mono && accept;
                accept = accept && !mono;
            }
            const unsigned long long mm = CRIT == 3 ? __ballot(mono) : 0ull;
            const unsigned long long am = __ballot(accept);
            const unsigned long long dm = __ballot(direct);
            const uint32_t nc = open ? meta_nchild(w.meta) : 0u;
            const uint32_t lc = direct ? meta_count(w.meta) : 0u;
            const uint32_t cinc = winclusive(nc);
            const uint32_t linc = winclusive(lc);
            int nm = static_cast<int>(__popcll(mm)), na = static_cast<int>(__popcll(am));
            int nd = static_cast<int>(__popcll(dm));
            int ctot = static_cast<int>(wlast(cinc));
            uint32_t ltot = wlast(linc);
            int om = 0, oa = 0, od = 0, oc = 0;
            uint32_t ol = 0;
            if (W > 1) {
                if (lane == 0) {
                    wtot[wv][0] = static_cast<uint32_t>(nm);
                    wtot[wv][1] = static_cast<uint32_t>(na) | (half_box ? kHalfBox : 0u);
                    wtot[wv][2] = static_cast<uint32_t>(nd);
                    wtot[wv][3] = static_cast<uint32_t>(ctot);
                    wtot[wv][4] = ltot;
                }
                __syncthreads();
                nm = na = nd = ctot = 0;
                ltot = 0;
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    const bool prior = k < wv;
                    om += prior ? static_cast<int>(wtot[k][0]) : 0;
                    const uint32_t nak = wtot[k][1];
                    far_image = far_image || (TPM && (nak & kHalfBox) != 0u);
                    oa += prior ? static_cast<int>(nak & ~kHalfBox) : 0;
                    od += prior ? static_cast<int>(wtot[k][2]) : 0;
                    oc += prior ? static_cast<int>(wtot[k][3]) : 0;
                    ol += prior ? wtot[k][4] : 0u;
                    nm += static_cast<int>(wtot[k][0]);
                    na += static_cast<int>(nak & ~kHalfBox);
                    nd += static_cast<int>(wtot[k][2]);
                    ctot += static_cast<int>(wtot[k][3]);
                    ltot += wtot[k][4];
                }
            }

            // 1) accepted nodes -> LDS cell list (point masses -> particle list)
            if (CRIT == 3 && nm > 0) {
                if (npart + nm >= kPartCap) {  // uniform; keeps npart < kPartCap
                    eval_parts<TPM, W>(pl, npart, j0, dj, far_image, tx, ty, tz, P, ax, ay, az);
                    npp += static_cast<unsigned long long>(npart);
                    npart = 0;
                    __syncthreads();
                }
                if (mono)
                    pl[npart + om + static_cast<int>(__popcll(mm & lt))] =
                        make_float4(px, py, pz, w.mass);
                npart += nm;
                nmono += static_cast<unsigned long long>(nm);
            }
            if (accept) {
                const int slot = ncell + oa + static_cast<int>(__popcll(am & lt));
                cl[slot].a = make_float4(px, py, pz, w.mass);
                // the open walk's expansion needs eps^2 trs, the TreePM one Q / 3, trs / 3
                // and 5/6 trs
                constexpr float third = 1.0f / 3.0f;
                if (TPM) {
                    cl[slot].b = make_float4(third * w.qxx, third * w.qxy, third * w.qxz,
                                             third * w.qyy);
                    cl[slot].c = make_float4(third * w.qyz, third * w.trs,
                                             -third * (w.qxx + w.qyy), (2.5f * third) * w.trs);
                } else {
                    cl[slot].b = make_float4(w.qxx, w.qxy, w.qxz, w.qyy);
                    cl[slot].c = make_float4(w.qyz, P.eps2 * w.trs, -(w.qxx + w.qyy), 0.0f);
                }
            }
            ncell += na;

            // 2) children of opened nodes -> traversal stack
            if (sp + ctot > stack_cap) {
                if (threadIdx.x == 0)
                    atomicOr(err, kErrStackOverflow);
            } else {
                const int base = sp + oc + static_cast<int>(cinc - nc);
                if (W == 1) {
                    if (open)
                        push_children(stk + base, w.first, nc);
                } else if (open) {
                    for (uint32_t j = 0; j < nc; ++j) {
                        const int at = base + static_cast<int>(j);
                        if (at < kLdsStack)
                            lstk[W > 1 ? at : 0] = w.first + static_cast<int>(j);
                        else
                            stk[at] = w.first + static_cast<int>(j);
                    }
                }
                sp += ctot;
            }

            // 3) opened leaves -> descriptors, then their particles -> LDS
            if (direct) {
                const int slot = od + static_cast<int>(__popcll(dm & lt));
                lfFirst[slot] = w.first;
                lfPre[slot] = ol + linc - lc;
                lfSx[slot] = sx;
                lfSy[slot] = sy;
                lfSz[slot] = sz;
            }
            if (static_cast<int>(threadIdx.x) >= nd)
                lfPre[threadIdx.x] = ~0u;  // past the last leaf, for the search below
            __syncthreads();

            if (FAR && nfl > kFarCap - 64) {
                far_flush(fl, nfl, nodes, rcx, rcy, rcz, ux, uy, uz, gcx, gcy, gcz, P.eps2, fsum);
                nfl = 0;
            }

            if (ncell > kCellCap - kThreads) {
                eval_cells<ORDER, TPM, W>(cl, ncell, j0, dj, far_image, tx, ty, tz, P, ax, ay, az);
                npc += static_cast<unsigned long long>(ncell);
                ncell = 0;
                __syncthreads();
            }

            uint32_t done = 0;
            const int top = nd > 1 ? 1 << (31 - __builtin_clz(static_cast<unsigned>(nd - 1))) : 0;
            while (done < ltot) {
                const uint32_t room = static_cast<uint32_t>(kPartCap - npart);
                const uint32_t chunk = ltot - done < room ? ltot - done : room;
                for (uint32_t f = threadIdx.x; f < chunk; f += static_cast<uint32_t>(kThreads)) {
                    const uint32_t gi = done + f;
                    // the last leaf that starts at gi or before: a step per bit of nd - 1,
                    // the same for all lanes, 3 VALU instructions each (7 with two bounds)
                    int lo = 0;
                    for (int step = top; step > 0; step >>= 1)
                        lo += lfPre[lo + step] <= gi ? step : 0;
                    const float4 q = spart[lfFirst[lo] + static_cast<int>(gi - lfPre[lo])];
                    pl[npart + static_cast<int>(f)] =
                        make_float4(q.x + lfSx[lo], q.y + lfSy[lo], q.z + lfSz[lo], q.w);
                }
                __syncthreads();
                npart += static_cast<int>(chunk);
                done += chunk;
                if (npart == kPartCap) {
                    eval_parts<TPM, W>(pl, npart, j0, dj, far_image, tx, ty, tz, P, ax, ay, az);
                    npp += static_cast<unsigned long long>(npart);
                    npart = 0;
                    __syncthreads();
                }
            }
        }
        eval_cells<ORDER, TPM, W>(cl, ncell, j0, dj, far_image, tx, ty, tz, P, ax, ay, az);
        eval_parts<TPM, W>(pl, npart, j0, dj, far_image, tx, ty, tz, P, ax, ay, az);
        npc += static_cast<unsigned long long>(ncell);
        npp += static_cast<unsigned long long>(npart);
        for (int o = 32; o >= tw; o >>= 1) {  // the list shares of one target
            ax += __shfl_xor(ax, o, 64);
            ay += __shfl_xor(ay, o, 64);
            az += __shfl_xor(az, o, 64);
        }
        if (W > 1) {
            // the waves' shares, in wave order (the lists are free now)
            __syncthreads();
            if (wv > 0)
                cl[(wv - 1) * 64 + lane].a = make_float4(ax, ay, az, 0.0f);
            __syncthreads();
            if (wv == 0) {
#pragma unroll
                for (int k = 0; k < W - 1; ++k) {
                    const float4 v = cl[k * 64 + lane].a;
                    ax += v.x;
                    ay += v.y;
                    az += v.z;
                }
            }
        }
        if (FAR) {
            // the rest of the queue, then the group's expansion at each target
            far_flush(fl, nfl, nodes, rcx, rcy, rcz, ux, uy, uz, gcx, gcy, gcz, P.eps2, fsum);
            nfl = 0;
            __syncthreads();
            float F[kFarTerms];
#pragma unroll
            for (int k = 0; k < kFarTerms; ++k)
                F[k] = fsum[k];
            far_evaluate(F, tx - gcx, ty - gcy, tz - gcz, ax, ay, az);
        }
        // per-target interaction counts for the roofline (only active lanes are real targets)
        npp = npp * static_cast<unsigned long long>(nact);
        npc = npc * static_cast<unsigned long long>(nact);
        tot_pp += npp;
        tot_pc += npc;
        if (CRIT == 3)
            tot_mono += nmono * static_cast<unsigned long long>(nact);
        if (FAR) {
            tot_far += nfar;                                      // node-group
            tot_eval += static_cast<unsigned long long>(nact);   // evaluations
        }
        npp = 0;
        npc = 0;
        if (REC && threadIdx.x == 0 && g < rec_groups)
            rec_n[g] = static_cast<uint32_t>(nrec < rec_cap ? nrec : rec_cap);
        __syncthreads();

        if (target && j0 == 0) {
            // OctHostMath.cpp:50-57
            const float mag = sqrtf(ax * ax + ay * ay + az * az);
            if (P.max_acc > 0.0f && mag > P.max_acc && mag > 1.0e-6f) {
                const float k = P.max_acc / mag;
                ax *= k;
                ay *= k;
                az *= k;
            }
            accx[s] = ax;
            accy[s] = ay;
            accz[s] = az;
            if (P.amag)
                P.amag[s] = sqrtf(ax * ax + ay * ay + az * az);
        }
    }
    if (stats && threadIdx.x == 0) {
        atomicAdd(&stats[0], tot_pp);
        atomicAdd(&stats[1], tot_pc);
        if (CRIT == 3 && tot_mono)
            atomicAdd(&stats[5], tot_mono);
        if (FAR) {
            atomicAdd(&stats[3], tot_far);
            atomicAdd(&stats[4], tot_eval);
        }
    }
}

// Waves per group. A walk keeps about `slots` waves resident (walk_slots, 24
// per CU). With fewer groups than that its time is the latency of its heaviest
// group, which W waves cut: they test 64 W nodes per step and split the lists.
// Past that point the chip is full and the steps' barriers only cost (2 waves
// per group: 5-20 % on the COM walk of 80,000 particles and more). Walk times
// in us with 1 / 2 / 4 / 8 waves (Plummer, theta 0.5; slots = 6,144):
//   COM, cap 16       4,099: 167 / 97 / 72 / 85     32,768: 394 / 278 / 262 / 398
//                    65,536: 600 / 561 / 588 / 906 100,003: 656 / 689 / 767 / -
//   bounds, cap 64   20,000: 979 / 513 / 378 / 221 100,000: 1284 / 941 / 759 / 906
//                   300,001: 2844 / 2550 / 2530 / 3154
//   relative        100,000: 374 / 286 / 296 / 616 260,000: 557 / 502 / 668 / -
//                   500,000: 578 / 587 / 756 / -
//   periodic TreePM  64^3:   492 / 450 / 541 / 881  128^3: 2250 / 2274 / 2505 / -
//   (with every pair's image rounded; 1 wave at 128^3 now 1990)
// The relative and TreePM walks, whose lists take longer per entry or flush
// more often, gain from 2 waves up to 3.5 groups per slot. COM runs keep one
// wave from 0.47 groups per slot on and under block time steps. That is a choice,
// no limit (against FP64 either order errs the same): adding a target's terms in
// another order moves its FP32 force by 2e-7 (4,096
// particles) to 5e-7 (65,536), which an FP64 state integrated over tens of steps
// shows (1.6e-9 of the velocities after 20 steps at 65,536), for 7 % of the walk
// there. The count depends on n, the criterion and the GPU only; the recording
// walk takes the plain one's, so that an idle correction changes no bit.
int walk_waves(const Device& d, const WalkParams& p)
{
    const float slots = static_cast<float>(d.walk_slots);
    const float G = static_cast<float>(walk_groups_usual(d.n, d.group_cap));
    if (p.alevel)
        return 1;
    if (p.criterion == 1 || p.criterion == 2)
        return 8.0f * G <= slots ? 8 : G <= 1.1f * slots ? 4 : 1;
    if (G <= kWalkFourWaves * slots)
        return 4;
    return (p.criterion == 3 || p.rs > 0.0f) && G <= 3.5f * slots ? 2 : 1;
}

template <int W, int ORDER, int CRIT, bool TPM, bool REC, bool FAR>
void launch_walk_w(Device& d, const WalkParams& p, unsigned long long* stats, const LffState* L,
                   float band, int min_count)
{
    // W waves per workgroup, each with a stack region. No more workgroups than
    // the groups n particles usually make (idle ones only draw tickets); nine
    // tenths of them with one wave each, where the light groups at the end of the
    // order fill in behind the heavy ones (COM walk at 67,657 particles, Plummer
    // / merger: n / 16 workgroups 633 / 414 us, n / 13 598 / 420, n / 11.5 614 / 445).
    const size_t usual = walk_groups_usual(d.n, d.group_cap);
    const unsigned grid = static_cast<unsigned>(std::max<size_t>(
        std::min(d.stack_waves / W, W == 1 ? usual - usual / 10 : usual), 1));
    walk_kernel<ORDER, CRIT, TPM, REC, FAR, W><<<grid, 64 * W, 0, d.stream>>>(
        p, d.wnode, d.spart, d.sleaf, d.geom, d.groups, d.level_info,
        static_cast<int>(d.node_cap), d.work_counter,
        d.stack, static_cast<int>(d.stack_cap), d.acc[0], d.acc[1], d.acc[2], d.err, stats,
        L ? L->lists : nullptr, L ? L->list_n : nullptr, L ? L->list_cap : 0,
        L ? static_cast<int>(L->list_groups) : 0, band * band,
        static_cast<uint32_t>(min_count > 0 ? min_count : 0));
}

template <int ORDER, int CRIT, bool TPM, bool REC = false, bool FAR = false>
void launch_walk_t(Device& d, const WalkParams& p, unsigned long long* stats,
                   const LffState* L = nullptr, float band = 0.0f, int min_count = 0)
{
    if constexpr (!FAR) {
        switch (walk_waves(d, p)) {
        case 8:
            if constexpr (CRIT == 1 || CRIT == 2)
                return launch_walk_w<8, ORDER, CRIT, TPM, REC, FAR>(d, p, stats, L, band, min_count);
            break;
        case 4:
            return launch_walk_w<4, ORDER, CRIT, TPM, REC, FAR>(d, p, stats, L, band, min_count);
        case 2:
            if constexpr (CRIT == 0 || CRIT == 3)
                return launch_walk_w<2, ORDER, CRIT, TPM, REC, FAR>(d, p, stats, L, band, min_count);
            break;
        default:
            break;
        }
    }
    launch_walk_w<1, ORDER, CRIT, TPM, REC, FAR>(d, p, stats, L, band, min_count);
}

}  // namespace

namespace {
void clear_tickets(Device& d)
{
    if (!d.tickets_zero)
        launch_fill_u32(d.work_counter, 0u, kTicketWords, d.stream);
    d.tickets_zero = false;  // the walk draws from them
}
}  // namespace

void launch_walk_record(Device& d, const WalkParams& p, unsigned long long* stats,
                        const LffState& L, float band, int min_count)
{
    if (d.n == 0)
        return;
    clear_tickets(d);
    if (p.criterion == 1)
        launch_walk_t<2, 1, false, true>(d, p, stats, &L, band, min_count);
    else if (p.criterion == 2)
        launch_walk_t<2, 2, false, true>(d, p, stats, &L, band, min_count);
    else
        launch_walk_t<2, 0, false, true>(d, p, stats, &L, band, min_count);
}

void launch_walk(Device& d, const WalkParams& p, unsigned long long* stats)
{
    if (d.n == 0)
        return;
    clear_tickets(d);
    const bool tpm = p.rs > 0.0f;
    if (p.far2 > 0.0f && !tpm && p.order >= 2) {
        // quadrupole walk with the group far-field expansion
        if (p.criterion == 1)
            launch_walk_t<2, 1, false, false, true>(d, p, stats);
        else if (p.criterion == 2)
            launch_walk_t<2, 2, false, false, true>(d, p, stats);
        else if (p.criterion == 3)
            launch_walk_t<2, 3, false, false, true>(d, p, stats);
        else
            launch_walk_t<2, 0, false, false, true>(d, p, stats);
        return;
    }
    if (p.criterion == 3) {
        if (p.order >= 2)
            tpm ? launch_walk_t<2, 3, true>(d, p, stats)
                : launch_walk_t<2, 3, false>(d, p, stats);
        else
            tpm ? launch_walk_t<1, 3, true>(d, p, stats)
                : launch_walk_t<1, 3, false>(d, p, stats);
    } else if (p.criterion == 2) {
        if (p.order >= 2)
            tpm ? launch_walk_t<2, 2, true>(d, p, stats)
                : launch_walk_t<2, 2, false>(d, p, stats);
        else
            tpm ? launch_walk_t<1, 2, true>(d, p, stats)
                : launch_walk_t<1, 2, false>(d, p, stats);
    } else if (p.order >= 2) {
        if (p.criterion == 1)
            tpm ? launch_walk_t<2, 1, true>(d, p, stats)
                : launch_walk_t<2, 1, false>(d, p, stats);
        else
            tpm ? launch_walk_t<2, 0, true>(d, p, stats)
                : launch_walk_t<2, 0, false>(d, p, stats);
    } else {
        if (p.criterion == 1)
            tpm ? launch_walk_t<1, 1, true>(d, p, stats)
                : launch_walk_t<1, 1, false>(d, p, stats);
        else
            tpm ? launch_walk_t<1, 0, true>(d, p, stats)
                : launch_walk_t<1, 0, false>(d, p, stats);
    }
}

}  // namespace bh
