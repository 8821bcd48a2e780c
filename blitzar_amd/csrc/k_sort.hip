// Stable sorts of (64-bit key, 32-bit value) pairs (tile sort and merge; LSD radix
// for large inputs), device-wide exclusive scan, equal-key tie ordering and the particle-store permutation.
//
// Contract followed: thrust::sort_by_key(keys, identity indices) at
// engine/physics/octree/cuda/linear/OctBuild.inl:96 -- ascending keys, equal
// keys keep ascending original particle index. The store is kept in the last
// sorted order, so the sort's own stability orders ties by previous slot;
// tie_fix_kernel then reorders every run of equal keys by particle id, which
// restores the reference contract exactly.
//
// One radix pass (8-bit digit) = histogram kernel (reads 8 B/key), one single-pass
// scan of the digit-major tile counts, and a scatter kernel that ranks keys inside a tile
// of 4096 with wave ballots, reorders the tile in LDS and writes digit runs
// contiguously (reads 12 B/key, writes 12 B/key).
#include "bh_internal.h"
#include "morton.h"
#include "scan_lookback.h"

namespace bh {
namespace {

constexpr int kBlock = 256;
#ifndef BH_SORT_ITEMS
#define BH_SORT_ITEMS 16
#endif
// Keys per thread. A tile of 4096 keys (16 per thread) writes digit runs of 16
// keys on average, twice those of a 2048-key tile: fewer partial cache lines
// (70 us less per 8M-key sort than 8 per thread, at 2 blocks per CU).
constexpr int kItems = BH_SORT_ITEMS;
constexpr int kTile = kBlock * kItems;  // keys per tile
constexpr int kWaves = kBlock / 64;

__device__ inline unsigned long long lanemask_lt()
{
    const unsigned lane = threadIdx.x & 63u;
    return lane == 0 ? 0ull : (~0ull >> (64u - lane));
}

__global__ __launch_bounds__(kBlock) void hist_kernel(const unsigned long long* __restrict__ keys,
                                                      size_t n, int shift, uint32_t dmask,
                                                      uint32_t* __restrict__ hist,
                                                      uint32_t ntiles)
{
    __shared__ uint32_t h[256];
    const int t = threadIdx.x;
    h[t] = 0;
    __syncthreads();
    const size_t base = static_cast<size_t>(blockIdx.x) * kTile;
    for (int k = 0; k < kItems; ++k) {
        const size_t i = base + static_cast<size_t>(k) * kBlock + t;
        if (i < n)
            atomicAdd(&h[(keys[i] >> shift) & dmask], 1u);
    }
    __syncthreads();
    hist[static_cast<size_t>(t) * ntiles + blockIdx.x] = h[t];
}

__global__ __launch_bounds__(kBlock) void scatter_kernel(
    const unsigned long long* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
    unsigned long long* __restrict__ keys_out, uint32_t* __restrict__ vals_out, size_t n,
    int shift, uint32_t dmask, const uint32_t* __restrict__ hist, uint32_t ntiles)
{
    __shared__ uint32_t wcnt[kWaves][256];
    __shared__ uint32_t tile_off[256];
    __shared__ uint32_t gbase[256];
    __shared__ uint32_t red[kWaves];
    __shared__ unsigned long long sk[kTile];
    __shared__ uint32_t sv[kTile];

    const int t = threadIdx.x;
    const int w = t >> 6;
    const int lane = t & 63;
    const size_t tile = blockIdx.x;
    const size_t tbase = tile * kTile;
    const uint32_t tile_n =
        static_cast<uint32_t>(n - tbase < static_cast<size_t>(kTile) ? n - tbase : kTile);

    for (int k = 0; k < kWaves; ++k)
        wcnt[k][t] = 0;
    gbase[t] = hist[static_cast<size_t>(t) * ntiles + tile];
    __syncthreads();

    unsigned long long key[kItems];
    uint32_t val[kItems];
    uint32_t rnk[kItems];
    const size_t wbase = tbase + static_cast<size_t>(w) * 64 * kItems;
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const size_t i = wbase + static_cast<size_t>(it) * 64 + lane;
        const bool valid = i < n;
        key[it] = valid ? keys_in[i] : 0ull;
        val[it] = valid ? vals_in[i] : 0u;
    }
    const unsigned long long lt = lanemask_lt();
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const size_t i = wbase + static_cast<size_t>(it) * 64 + lane;
        const bool valid = i < n;
        const uint32_t d = static_cast<uint32_t>(key[it] >> shift) & dmask;
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const unsigned long long m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t before = static_cast<uint32_t>(__popcll(peers & lt));
        const uint32_t base = valid ? wcnt[w][d] : 0u;
        // The lowest lane of each digit group advances that wave's counter;
        // LDS operations of one wave complete in program order, so every
        // lane has read the old value above.
        if (valid && before == 0)
            wcnt[w][d] = base + static_cast<uint32_t>(__popcll(peers));
        rnk[it] = base + before;
    }
    __syncthreads();
    // Per digit: exclusive offsets across waves, then across digits in the tile.
    {
        uint32_t run = 0;
        for (int k = 0; k < kWaves; ++k) {
            const uint32_t c = wcnt[k][t];
            wcnt[k][t] = run;
            run += c;
        }
        uint32_t total;
        const uint32_t ex = block_exclusive256(run, red, &total);
        tile_off[t] = ex;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const size_t i = wbase + static_cast<size_t>(it) * 64 + lane;
        if (i < n) {
            const uint32_t d = static_cast<uint32_t>(key[it] >> shift) & dmask;
            const uint32_t pos = tile_off[d] + wcnt[w][d] + rnk[it];
            sk[pos] = key[it];
            sv[pos] = val[it];
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kItems; ++m) {
        const uint32_t j = static_cast<uint32_t>(m) * kBlock + t;
        if (j < tile_n) {
            const unsigned long long k = sk[j];
            const uint32_t d = static_cast<uint32_t>(k >> shift) & dmask;
            const size_t out = static_cast<size_t>(gbase[d]) + (j - tile_off[d]);
            keys_out[out] = k;
            vals_out[out] = sv[j];
        }
    }
}

// ---- device-wide exclusive scan (element count from host or device) -------
__global__ __launch_bounds__(kScanBlock) void scan_lookback_kernel(
    uint32_t* __restrict__ data, const int* n_dev, size_t n_host, uint32_t* __restrict__ ws,
    uint32_t* total_out, int* total_out_i, int* err)
{
    size_t n = n_dev ? static_cast<size_t>(*n_dev > 0 ? *n_dev : 0) : n_host;
    n = n < static_cast<size_t>(gridDim.x) * kScanChunk ? n : static_cast<size_t>(gridDim.x) * kScanChunk;
    const ScanBlockResult r = scan_lookback_block(data, n, ws, err, kErrScan);
    if (r.last && threadIdx.x == 0) {
        if (total_out)
            *total_out = r.total;
        if (total_out_i)
            *total_out_i = static_cast<int>(r.total);
    }
}

// ---- tile sort and merge ----------------------------------------------------
// Tiles are sorted in LDS by merging (8 pairs per thread in registers, then
// runs two by two), and the tiles' runs are merged two by two in memory (merge
// path). Everything is stable. FULL: keys compare whole; else under kmask.
// Bound: latency up to a few hundred thousand pairs (a tile of 4,096: 9 rounds of
// a binary search and 8 dependent LDS reads, 26 us; a merge pass 8-10 us, half of
// it the split search), then the merge's issue rate (2,097,152 pairs: 17 us a pass,
// 2.9 TB/s). Sorting the tiles with the radix sort's ballot ranking took 39 us.
constexpr int kMergePer = 8;  // pairs per thread

// LDS place of pair i: one unused place after every 8, so that threads 8 pairs
// apart meet different banks.
__host__ __device__ constexpr uint32_t lds_at(uint32_t i) { return i + (i >> 3); }

template <bool FULL>
__device__ inline bool key_gt(unsigned long long a, unsigned long long b, unsigned long long kmask)
{
    return FULL ? a > b : (a & kmask) > (b & kmask);
}

// First kMergePer outputs from output dd on of the merge of A = sk[a, a + na) and
// B = sk[b, b + nb) (equal keys: A first), in registers; dd <= na + nb, outputs past
// na + nb are not defined.
template <bool FULL>
__device__ inline void lds_merge(const unsigned long long* sk, const uint32_t* sv, uint32_t a,
                                 uint32_t na, uint32_t b, uint32_t nb, uint32_t dd,
                                 unsigned long long kmask, unsigned long long* key, uint32_t* val)
{
    uint32_t lo = dd > nb ? dd - nb : 0u, hi = dd < na ? dd : na;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (key_gt<FULL>(sk[lds_at(a + mid)], sk[lds_at(b + dd - 1u - mid)], kmask))
            hi = mid;
        else
            lo = mid + 1u;
    }
    uint32_t ia = a + lo, ib = b + dd - lo;
    const uint32_t ea = a + na, eb = b + nb;
    unsigned long long ka = ia < ea ? sk[lds_at(ia)] : 0ull,
                       kb = ib < eb ? sk[lds_at(ib)] : 0ull;
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        const bool ta = ia < ea && (ib >= eb || !key_gt<FULL>(ka, kb, kmask));
        key[k] = ta ? ka : kb;
        const uint32_t at = ta ? ia : ib;
        val[k] = at < eb ? sv[lds_at(at)] : 0u;
        ia += ta ? 1u : 0u;
        ib += ta ? 0u : 1u;
        const uint32_t nx = ta ? ia : ib;
        const unsigned long long kn = nx < (ta ? ea : eb) ? sk[lds_at(nx)] : 0ull;
        ka = ta ? kn : ka;
        kb = ta ? kb : kn;
    }
}

// Sorts THREADS * kMergePer pairs in sk / sv (places past the valid pairs hold
// keys of all ones, which stay behind every valid pair). Every thread calls it
// after a barrier; it ends with one.
template <int THREADS, bool FULL>
__device__ inline void tile_sort(unsigned long long* sk, uint32_t* sv, unsigned long long kmask)
{
    const uint32_t o = threadIdx.x * kMergePer;
    unsigned long long key[kMergePer];
    uint32_t val[kMergePer];
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        key[k] = sk[lds_at(o + k)];
        val[k] = sv[lds_at(o + k)];
    }
    // odd-even transposition: neighbours swap only when out of order
#pragma unroll
    for (int r = 0; r < kMergePer; ++r)
#pragma unroll
        for (int k = r & 1; k + 1 < kMergePer; k += 2) {
            const bool sw = key_gt<FULL>(key[k], key[k + 1], kmask);
            const unsigned long long x = key[k], y = key[k + 1];
            const uint32_t u = val[k], v = val[k + 1];
            key[k] = sw ? y : x;
            key[k + 1] = sw ? x : y;
            val[k] = sw ? v : u;
            val[k + 1] = sw ? u : v;
        }
#pragma unroll 1
    for (uint32_t run = kMergePer;; run *= 2) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kMergePer; ++k) {
            sk[lds_at(o + k)] = key[k];
            sv[lds_at(o + k)] = val[k];
        }
        __syncthreads();
        if (run >= THREADS * kMergePer)
            return;
        const uint32_t p = o & ~(2u * run - 1u);
        lds_merge<FULL>(sk, sv, p, run, p + run, run, o - p, kmask, key, val);
    }
}

// Where a tile's pairs come from: arrays, or the particles' positions (MODE 0 or
// 1: the key mode; the value is the store slot).
struct PairsIn {
    const unsigned long long* __restrict__ keys;
    const uint32_t* __restrict__ vals;
    __device__ void load(size_t i, unsigned long long& k, uint32_t& v) const
    {
        k = keys[i];
        v = vals[i];
    }
};
template <int MODE>
struct PositionsIn {
    const double* __restrict__ px;
    const double* __restrict__ py;
    const double* __restrict__ pz;
    const RootGeom* __restrict__ g;
    __device__ void load(size_t i, unsigned long long& k, uint32_t& v) const
    {
        k = morton_key<MODE>(px[i], py[i], pz[i], g);
        v = static_cast<uint32_t>(i);
    }
};

template <int THREADS, bool FULL, class In>
__global__ __launch_bounds__(THREADS) void tile_sort_kernel(
    In in, unsigned long long* __restrict__ keys_out, uint32_t* __restrict__ vals_out, size_t n,
    unsigned long long kmask)
{
    constexpr uint32_t T = THREADS * kMergePer;
    __shared__ unsigned long long sk[lds_at(T)];
    __shared__ uint32_t sv[lds_at(T)];
    const size_t t0 = static_cast<size_t>(blockIdx.x) * T;
    const uint32_t tn = static_cast<uint32_t>(n - t0 < T ? n - t0 : T);
    unsigned long long key[kMergePer];
    uint32_t val[kMergePer];
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        const uint32_t i = threadIdx.x + k * THREADS;
        key[k] = ~0ull;
        val[k] = 0u;
        if (i < tn)
            in.load(t0 + i, key[k], val[k]);
    }
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        const uint32_t i = threadIdx.x + k * THREADS;
        sk[lds_at(i)] = key[k];
        sv[lds_at(i)] = val[k];
    }
    __syncthreads();
    tile_sort<THREADS, FULL>(sk, sv, kmask);
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        const uint32_t i = threadIdx.x + k * THREADS;
        if (i < tn) {
            keys_out[t0 + i] = sk[lds_at(i)];
            vals_out[t0 + i] = sv[lds_at(i)];
        }
    }
}

// Elements of A among the first d of the merge of A[0, la) and B[0, lb) (equal
// keys: A first), by a whole wavefront: 64 probes per step, each step one round
// trip for a 64th of the range.
template <bool FULL>
__device__ inline uint32_t wave_merge_split(const unsigned long long* __restrict__ A, uint32_t la,
                                            const unsigned long long* __restrict__ B, uint32_t lb,
                                            uint32_t d, unsigned long long kmask)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lo = d > lb ? d - lb : 0u, hi = d < la ? d : la;
    while (lo < hi) {  // the first i in [lo, hi) with A[i] > B[d - 1 - i], else hi
        const uint32_t step = (hi - lo + 63u) / 64u;
        const uint32_t i = lo + lane * step;
        const bool past = i >= hi || key_gt<FULL>(A[i], B[d - 1u - i], kmask);
        const unsigned long long m = __ballot(past);
        const uint32_t f = m ? static_cast<uint32_t>(__builtin_ctzll(m)) : 64u;
        if (f == 0u)
            break;  // already past at lo
        const uint32_t at = lo + f * step;
        lo += (f - 1u) * step + 1u;
        hi = at < hi ? at : hi;
    }
    return lo;
}

// One merge pass: runs of `run` pairs (a multiple of kMergeOut / 2, the last
// one ragged) two by two into runs of 2 run; a block writes kMergeOut
// consecutive pairs of one merged run.
constexpr int kMergeBlock = 256;
constexpr int kMergeOut = kMergeBlock * kMergePer;

template <bool FULL>
__global__ __launch_bounds__(kMergeBlock) void merge_kernel(
    const unsigned long long* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
    unsigned long long* __restrict__ keys_out, uint32_t* __restrict__ vals_out, size_t n,
    size_t run, unsigned long long kmask)
{
    __shared__ unsigned long long sk[lds_at(kMergeOut)];
    __shared__ uint32_t sv[lds_at(kMergeOut)];
    __shared__ uint32_t split[2];
    const int t = threadIdx.x;
    const size_t o0 = static_cast<size_t>(blockIdx.x) * kMergeOut;
    const size_t p0 = o0 / (2 * run) * (2 * run);
    const uint32_t la = static_cast<uint32_t>(n - p0 < run ? n - p0 : run);
    const uint32_t lb =
        static_cast<uint32_t>(n - p0 - la < run ? n - p0 - la : run);
    const unsigned long long* A = keys_in + p0;
    const unsigned long long* B = A + la;
    const uint32_t d0 = static_cast<uint32_t>(o0 - p0);
    const uint32_t d1 = d0 + kMergeOut < la + lb ? d0 + kMergeOut : la + lb;
    const uint32_t cnt = d1 - d0;
    if (t < 128) {
        const uint32_t v = wave_merge_split<FULL>(A, la, B, lb, t < 64 ? d0 : d1, kmask);
        if ((t & 63) == 0)
            split[t >> 6] = v;
    }
    __syncthreads();
    const uint32_t a0 = split[0], a1 = split[1];
    const uint32_t na = a1 - a0, nb = cnt - na;
    // outputs d0.. take A[a0, a1) and B[d0 - a0, ...): i < na from A, else from B
    const size_t ga = p0 + a0, gb = p0 + la + (d0 - a0) - na;
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        const uint32_t i = static_cast<uint32_t>(t + k * kMergeBlock);
        if (i < cnt) {
            const size_t g = (i < na ? ga : gb) + i;
            sk[lds_at(i)] = keys_in[g];
            sv[lds_at(i)] = vals_in[g];
        }
    }
    __syncthreads();
    const uint32_t o = static_cast<uint32_t>(t * kMergePer);
    unsigned long long key[kMergePer];
    uint32_t val[kMergePer];
    lds_merge<FULL>(sk, sv, 0u, na, na, nb, o < cnt ? o : cnt, kmask, key, val);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMergePer; ++k)
        if (o + k < cnt) {
            sk[lds_at(o + k)] = key[k];
            sv[lds_at(o + k)] = val[k];
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMergePer; ++k) {
        const uint32_t i = static_cast<uint32_t>(t + k * kMergeBlock);
        if (i < cnt) {
            keys_out[o0 + i] = sk[lds_at(i)];
            vals_out[o0 + i] = sv[lds_at(i)];
        }
    }
}

// Runs of equal keys: order the run by particle id (insertion sort; runs are
// short unless particles coincide).
__global__ __launch_bounds__(256) void tie_fix_kernel(const unsigned long long* __restrict__ keys,
                                                      uint32_t* __restrict__ vals,
                                                      const uint32_t* __restrict__ id, size_t n)
{
    const size_t s = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s + 1 >= n)
        return;
    const unsigned long long k = keys[s];
    if (keys[s + 1] != k || (s > 0 && keys[s - 1] == k))
        return;
    size_t e = s + 2;
    while (e < n && keys[e] == k)
        ++e;
    for (size_t a = s + 1; a < e; ++a) {
        const uint32_t v = vals[a];
        const uint32_t key_id = id[v];
        size_t b = a;
        while (b > s && id[vals[b - 1]] > key_id) {
            vals[b] = vals[b - 1];
            --b;
        }
        vals[b] = v;
    }
}

// The store follows the sort in two parts. Positions and masses, which the
// moments need, go first on the build's main stream; velocities, ids and the
// relative criterion's |a|, needed only by the walk and the integrator, go
// on the second stream beside the moments.
__global__ __launch_bounds__(256) void permute_store_kernel(
    const uint32_t* __restrict__ src, size_t n, const double* __restrict__ px,
    const double* __restrict__ py, const double* __restrict__ pz, const float* __restrict__ m,
    double* __restrict__ opx, double* __restrict__ opy, double* __restrict__ opz,
    float* __restrict__ om)
{
    const size_t s = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    const uint32_t j = src[s];
    opx[s] = px[j];
    opy[s] = py[j];
    opz[s] = pz[j];
    om[s] = m[j];
}

__global__ __launch_bounds__(256) void permute_rest_kernel(
    const uint32_t* __restrict__ src, size_t n, const double* __restrict__ vx,
    const double* __restrict__ vy, const double* __restrict__ vz,
    const uint32_t* __restrict__ id, const float* __restrict__ am, double* __restrict__ ovx,
    double* __restrict__ ovy, double* __restrict__ ovz, uint32_t* __restrict__ oid,
    float* __restrict__ oam)
{
    const size_t s = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    const uint32_t j = src[s];
    ovx[s] = vx[j];
    ovy[s] = vy[j];
    ovz[s] = vz[j];
    oid[s] = id[j];
    if (am)
        oam[s] = am[j];
}

// Both parts in one launch, where they run one after the other anyway. It also orders
// equal keys by particle id (tie_fix_kernel's launch, 4 us of a small build's 170): the
// thread at place s moves its source to the run's start plus the ids of the run below
// its own. src_out takes the fixed order.
__global__ __launch_bounds__(256) void permute_all_kernel(
    const unsigned long long* __restrict__ keys, const uint32_t* __restrict__ src,
    uint32_t* __restrict__ src_out, size_t n, const double* __restrict__ px,
    const double* __restrict__ py, const double* __restrict__ pz, const float* __restrict__ m,
    const double* __restrict__ vx, const double* __restrict__ vy, const double* __restrict__ vz,
    const uint32_t* __restrict__ id, const float* __restrict__ am, double* __restrict__ opx,
    double* __restrict__ opy, double* __restrict__ opz, float* __restrict__ om,
    double* __restrict__ ovx, double* __restrict__ ovy, double* __restrict__ ovz,
    uint32_t* __restrict__ oid, float* __restrict__ oam)
{
    size_t s = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    const uint32_t j = src[s];
    const uint32_t jid = id[j];
    const unsigned long long k = keys[s];
    if ((s > 0 && keys[s - 1] == k) || (s + 1 < n && keys[s + 1] == k)) {
        size_t at = s, below = 0;
        for (; at > 0 && keys[at - 1] == k; --at)
            below += id[src[at - 1]] < jid ? 1 : 0;
        for (size_t e = s + 1; e < n && keys[e] == k; ++e)
            below += id[src[e]] < jid ? 1 : 0;
        s = at + below;
    }
    src_out[s] = j;
    opx[s] = px[j];
    opy[s] = py[j];
    opz[s] = pz[j];
    om[s] = m[j];
    ovx[s] = vx[j];
    ovy[s] = vy[j];
    ovz[s] = vz[j];
    oid[s] = jid;
    if (am)
        oam[s] = am[j];
}

// The block time-step arrays follow the store through the same permutation.
__global__ __launch_bounds__(256) void permute_adaptive_kernel(
    const uint32_t* __restrict__ src, size_t n, const float* __restrict__ ax,
    const float* __restrict__ ay, const float* __restrict__ az, const uint32_t* __restrict__ lv,
    const uint32_t* __restrict__ lt, float* __restrict__ oax, float* __restrict__ oay,
    float* __restrict__ oaz, uint32_t* __restrict__ olv, uint32_t* __restrict__ olt)
{
    const size_t s = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    const uint32_t j = src[s];
    oax[s] = ax[j];
    oay[s] = ay[j];
    oaz[s] = az[j];
    olv[s] = lv[j];
    olt[s] = lt[j];
}

// rank[id[s]] = s: caller index -> store slot (rebuilt only when an API call
// needs it, not every step).
__global__ __launch_bounds__(256) void rank_kernel(const uint32_t* __restrict__ id, size_t n,
                                                   uint32_t* __restrict__ rank)
{
    const size_t s = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s < n)
        rank[id[s]] = static_cast<uint32_t>(s);
}

__global__ void fill_u32_kernel(uint32_t* p, uint32_t v, size_t n)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = v;
}

__global__ void begin_call_kernel(int* err, unsigned long long* stats)
{
    if (threadIdx.x == 0)
        *err = 0;
    if (threadIdx.x < 8)
        stats[threadIdx.x] = 0ull;
}

__global__ __launch_bounds__(256) void end_build_kernel(const int* err, EndBuild end)
{
    end_build(err, end);
}

__global__ void report_kernel(const int* err, const unsigned long long* stats, const int* info,
                              HostReport* rep)
{
    if (threadIdx.x == 0)
        rep->err = *err;
    if (threadIdx.x < 8)
        rep->stats[threadIdx.x] = stats[threadIdx.x];
    if (threadIdx.x < 2 * kLevels + 4)
        rep->info[threadIdx.x] = info[threadIdx.x];
}

}  // namespace

size_t scan_block_sums_words(size_t max_n) { return scan_workspace_words(max_n); }

void launch_scan_exclusive(uint32_t* data, size_t max_n, const int* n_dev, size_t n_host,
                           uint32_t* block_sums, uint32_t* total_out, int* total_out_i,
                           int* err, hipStream_t s)
{
    const size_t cap = n_dev ? max_n : n_host;
    const unsigned nb = static_cast<unsigned>(std::max<size_t>(1, (cap + kScanChunk - 1) / kScanChunk));
    scan_lookback_kernel<<<nb, kScanBlock, 0, s>>>(data, n_dev, n_host, block_sums, total_out,
                                                   total_out_i, err);
}

size_t radix_hist_words(size_t n)
{
    const size_t tiles = std::max<size_t>(1, (n + kTile - 1) / kTile);
    return 256 * tiles + scan_block_sums_words(256 * tiles);
}

namespace {

// Tile sort and merge, or LSD radix? The radix sort's time is its passes' (20 us
// each up to 65,536 pairs: three launches that leave the chip idle; 84 us at
// 8,388,608), whatever their order; the merge sort adds a pass per doubling of
// n past the tile. Sorts inside a build, us, merge / radix: 4,099 pairs 38 / 140,
// 65,536 64 / 182, 1,048,576 128 / 212, 4,194,304 370 / 416, 8,388,608
// 750 / 672. With 4 passes (30-bit keys) they meet near 131,072 pairs (110 / 114).
bool use_merge(size_t n, int key_bits)
{
    const int passes = (key_bits + 7) / 8;
    return passes > 1 && n <= (static_cast<size_t>(4096) << (5 * passes / 4));
}

// Threads of a tile's workgroup (8 pairs each). A tile is one workgroup's latency,
// 2.5 us per doubling with 512 threads, 4 with 1,024: the larger tile pays once
// it saves a pass over many pairs (2,097,152: 187 / 179 us).
int tile_threads(size_t n) { return n <= 2048 ? 256 : n <= 1200000 ? 512 : 1024; }

// Returns true when the result is in the first output pair. Reads `in` only in the
// first pass.
template <bool FULL, class In>
bool merge_sort(const In& in, unsigned long long* kout, uint32_t* vout, unsigned long long* knext,
                uint32_t* vnext, size_t n, unsigned long long kmask, hipStream_t stream)
{
    const int threads = tile_threads(n);
    const size_t tile = static_cast<size_t>(threads) * kMergePer;
    const unsigned nt = static_cast<unsigned>((n + tile - 1) / tile);
    if (threads == 256)
        tile_sort_kernel<256, FULL><<<nt, 256, 0, stream>>>(in, kout, vout, n, kmask);
    else if (threads == 512)
        tile_sort_kernel<512, FULL><<<nt, 512, 0, stream>>>(in, kout, vout, n, kmask);
    else
        tile_sort_kernel<1024, FULL><<<nt, 1024, 0, stream>>>(in, kout, vout, n, kmask);
    const unsigned nb = static_cast<unsigned>((n + kMergeOut - 1) / kMergeOut);
    bool first = true;
    for (size_t run = tile; run < n; run *= 2) {
        merge_kernel<FULL><<<nb, kMergeBlock, 0, stream>>>(kout, vout, knext, vnext, n, run, kmask);
        std::swap(kout, knext);
        std::swap(vout, vnext);
        first = !first;
    }
    return first;
}

}  // namespace

int radix_sort_passes(size_t n, int key_bits)
{
    if (!use_merge(n, key_bits))
        return (key_bits + 7) / 8;
    int passes = 1;  // the tiles
    for (size_t run = static_cast<size_t>(tile_threads(n)) * kMergePer; run < n; run *= 2)
        ++passes;
    return passes;
}

bool sort_uses_scan(size_t n, int key_bits) { return !use_merge(n, key_bits); }

bool radix_sort_from(const uint64_t* keys_in, const uint32_t* vals_in, uint64_t* keys_a,
                     uint32_t* vals_a, uint64_t* keys_b, uint32_t* vals_b, uint32_t* hist_ws,
                     size_t n, int key_bits, int* err, hipStream_t stream)
{
    const int passes = radix_sort_passes(n, key_bits);
    if (n <= 1)
        return false;
    if (use_merge(n, key_bits)) {
        const PairsIn in{reinterpret_cast<const unsigned long long*>(keys_in), vals_in};
        unsigned long long* ka = reinterpret_cast<unsigned long long*>(keys_a);
        unsigned long long* kb = reinterpret_cast<unsigned long long*>(keys_b);
        return key_bits < 64 ? merge_sort<false>(in, ka, vals_a, kb, vals_b, n,
                                                 (1ull << key_bits) - 1ull, stream)
                             : merge_sort<true>(in, ka, vals_a, kb, vals_b, n, ~0ull, stream);
    }
    const uint32_t ntiles = static_cast<uint32_t>((n + kTile - 1) / kTile);
    const size_t hn = static_cast<size_t>(ntiles) * 256;
    uint32_t* hist = hist_ws;
    uint32_t* sums = hist_ws + hn;
    const unsigned long long* kin = reinterpret_cast<const unsigned long long*>(keys_in);
    const uint32_t* vin = vals_in;
    unsigned long long* kout = reinterpret_cast<unsigned long long*>(keys_a);
    uint32_t* vout = vals_a;
    unsigned long long* knext = reinterpret_cast<unsigned long long*>(keys_b);
    uint32_t* vnext = vals_b;
    for (int p = 0; p < passes; ++p) {
        const int shift = 8 * p;
        // The last digit covers only the remaining key bits.
        const int bits = key_bits - shift < 8 ? key_bits - shift : 8;
        const uint32_t dmask = (1u << bits) - 1u;
        hist_kernel<<<ntiles, kBlock, 0, stream>>>(kin, n, shift, dmask, hist, ntiles);
        launch_scan_exclusive(hist, hn, nullptr, hn, sums, nullptr, nullptr, err, stream);
        scatter_kernel<<<ntiles, kBlock, 0, stream>>>(kin, vin, kout, vout, n, shift, dmask,
                                                      hist, ntiles);
        // this pass's output is the next pass's input; the next output is the
        // other buffer pair
        kin = kout;
        vin = vout;
        std::swap(kout, knext);
        std::swap(vout, vnext);
    }
    return (passes & 1) != 0;
}

bool radix_sort_buffers(uint64_t* keys, uint64_t* keys_alt, uint32_t* vals, uint32_t* vals_alt,
                        uint32_t* hist_ws, size_t n, int key_bits, int* err, hipStream_t stream)
{
    return radix_sort_from(keys, vals, keys_alt, vals_alt, keys, vals, hist_ws, n, key_bits, err,
                           stream);
}

void launch_radix_sort(Device& d, size_t n, int key_bits)
{
    if (n <= 1)
        return;
    if (radix_sort_buffers(d.keys, d.keys_b, d.vals, d.vals_b, d.sort_hist, n, key_bits, d.err,
                           d.stream)) {
        // Result is in the alternate buffers: swap the roles so d.keys/d.vals hold it.
        std::swap(d.keys, d.keys_b);
        std::swap(d.vals, d.vals_b);
    }
}

bool use_keys_sort(size_t n, int key_mode) { return n > 1 && use_merge(n, key_mode == 1 ? 30 : 63); }

void launch_keys_sort(Device& d, int key_mode)
{
    // keys end in d.keys_b / d.vals_b when the first output pair holds them
    unsigned long long* ka = reinterpret_cast<unsigned long long*>(d.keys_b);
    unsigned long long* kb = reinterpret_cast<unsigned long long*>(d.keys);
    // (63- and 30-bit keys hold nothing above those bits: they compare whole)
    const bool first =
        key_mode == 1
            ? merge_sort<true>(PositionsIn<1>{d.pos[0], d.pos[1], d.pos[2], d.geom}, ka, d.vals_b,
                               kb, d.vals, d.n, ~0ull, d.stream)
            : merge_sort<true>(PositionsIn<0>{d.pos[0], d.pos[1], d.pos[2], d.geom}, ka, d.vals_b,
                               kb, d.vals, d.n, ~0ull, d.stream);
    if (first) {
        std::swap(d.keys, d.keys_b);
        std::swap(d.vals, d.vals_b);
    }
}

void launch_tie_fix(Device& d)
{
    if (d.n < 2)
        return;
    const unsigned blocks = static_cast<unsigned>((d.n + 255) / 256);
    tie_fix_kernel<<<blocks, 256, 0, d.stream>>>(reinterpret_cast<const unsigned long long*>(d.keys),
                                                d.vals, d.id, d.n);
}

namespace {

void swap_positions(Device& d)
{
    for (int a = 0; a < 3; ++a)
        std::swap(d.pos[a], d.pos_b[a]);
    std::swap(d.mass, d.mass_b);
}

void swap_rest(Device& d)
{
    for (int a = 0; a < 3; ++a)
        std::swap(d.vel[a], d.vel_b[a]);
    std::swap(d.id, d.id_b);
    if (d.amag_live)
        std::swap(d.amag, d.amag_b);
}

void permute_adaptive(Device& d, unsigned blocks, hipStream_t st)
{
    if (!d.alevel)
        return;
    permute_adaptive_kernel<<<blocks, 256, 0, st>>>(
        d.vals, d.n, d.aacc[0], d.aacc[1], d.aacc[2], d.alevel, d.atick, d.aacc_b[0], d.aacc_b[1],
        d.aacc_b[2], d.alevel_b, d.atick_b);
    for (int a = 0; a < 3; ++a)
        std::swap(d.aacc[a], d.aacc_b[a]);
    std::swap(d.alevel, d.alevel_b);
    std::swap(d.atick, d.atick_b);
}

}  // namespace

void launch_permute_store(Device& d, hipStream_t st)
{
    if (d.n == 0)
        return;
    const unsigned blocks = static_cast<unsigned>((d.n + 255) / 256);
    permute_store_kernel<<<blocks, 256, 0, st>>>(d.vals, d.n, d.pos[0], d.pos[1], d.pos[2],
                                                 d.mass, d.pos_b[0], d.pos_b[1], d.pos_b[2],
                                                 d.mass_b);
    swap_positions(d);
}

void launch_permute_rest(Device& d, hipStream_t st)
{
    if (d.n == 0)
        return;
    const unsigned blocks = static_cast<unsigned>((d.n + 255) / 256);
    permute_rest_kernel<<<blocks, 256, 0, st>>>(
        d.vals, d.n, d.vel[0], d.vel[1], d.vel[2], d.id, d.amag_live ? d.amag : nullptr,
        d.vel_b[0], d.vel_b[1], d.vel_b[2], d.id_b, d.amag_b);
    swap_rest(d);
    permute_adaptive(d, blocks, st);
}

void launch_permute_all(Device& d, hipStream_t st)
{
    if (d.n == 0)
        return;
    const unsigned blocks = static_cast<unsigned>((d.n + 255) / 256);
    permute_all_kernel<<<blocks, 256, 0, st>>>(
        reinterpret_cast<const unsigned long long*>(d.keys), d.vals, d.vals_b, d.n, d.pos[0], d.pos[1], d.pos[2], d.mass, d.vel[0], d.vel[1], d.vel[2], d.id,
        d.amag_live ? d.amag : nullptr, d.pos_b[0], d.pos_b[1], d.pos_b[2], d.mass_b, d.vel_b[0],
        d.vel_b[1], d.vel_b[2], d.id_b, d.amag_b);
    std::swap(d.vals, d.vals_b);
    swap_positions(d);
    swap_rest(d);
    permute_adaptive(d, blocks, st);
}

void launch_rank(Device& d)
{
    if (d.n == 0)
        return;
    rank_kernel<<<static_cast<unsigned>((d.n + 255) / 256), 256, 0, d.stream>>>(d.id, d.n, d.rank);
}

void launch_begin_call(Device& d, unsigned long long* stats)
{
    begin_call_kernel<<<1, 64, 0, d.stream>>>(d.err, stats);
}

void launch_end_build(Device& d)
{
    end_build_kernel<<<1, 256, 0, d.stream>>>(d.err, EndBuild{d.work_counter, d.report});
    d.tickets_zero = true;
}

void launch_report(Device& d, const unsigned long long* stats)
{
    report_kernel<<<1, 64, 0, d.stream>>>(d.err, stats, d.level_info, d.report);
}

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s)
{
    if (n == 0)
        return;
    fill_u32_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(p, v, n);
}

}  // namespace bh
