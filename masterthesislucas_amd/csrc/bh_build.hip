// Tree build of the Barnes-Hut force step on gfx950:
//   bounds -> Morton codes -> sort -> gather into sorted SoA ->
//   leaf levels -> node count scan -> pre-order node emission -> upward mass/COM/M2 pass.
//
// The tree is laid out in pre-order over Morton-sorted particles: every node covers a
// contiguous particle range, its first child (if any) is the next node, and `skip` points past
// its subtree. Nodes starting at sorted index i are the cells of levels
// lcp(i-1, i)+1 .. leaf_level(i) whose first particle is i, so the layout follows from one scan.
//
// No kernel here uses device-scope fences, and same-address device atomics only to hand out the tiles
// of a sort: on a multi-XCD part both are expensive (a device-scope fence writes back or invalidates
// the XCD's L2). Results pass between kernels, and within a kernel through LDS; the exception are the
// sorts' look-back words, each a state and a count in one relaxed device-scope word that needs no
// fence.
#include "bh_common.h"
#include "bh_launch.h"

namespace bh {

// ------------------------------------------------------------------------------------------
// bounds: FP32 min/max per block, then one block derives the root square and the quantiser
// ------------------------------------------------------------------------------------------
// status word 1: the build saw a non-finite position (read by the host after the build)
__device__ __forceinline__ void flag_nonfinite(float4 r, uint32_t* status) {
    if (!(isfinite(r.x) && isfinite(r.y) && isfinite(r.z) && isfinite(r.w))) status[1] = 1u;
}

__global__ __launch_bounds__(kBlock) void k_bounds_partial(const float* __restrict__ xs,
                                                           const float* __restrict__ ys,
                                                           uint32_t n,
                                                           float4* __restrict__ partials) {
    float4 r = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        r = minmax4(r, bounds_item(xs[i], ys[i]));
    r = block_minmax4(r);
    if (threadIdx.x == 0) partials[blockIdx.x] = r;
}

__device__ void fill_params(BuildParams* prm, float4 r, uint64_t mnx64, uint64_t mny64,
                            uint64_t mxx64, uint64_t mxy64, uint32_t tree_mode, uint32_t n);

// the caller's bounds, or none
struct CallerBounds {
    int use;
    double minx, miny, maxx, maxy;
};

// every thread of the block takes part; thread 0 fills *out (LDS or memory). Without partials (nb =
// 0) the block takes the bounds of all positions itself.
__device__ __forceinline__ void bounds_final(const float4* __restrict__ partials, uint32_t nb,
                                             const float* __restrict__ xs,
                                             const float* __restrict__ ys, uint32_t n,
                                             uint32_t tree_mode, CallerBounds cb, BuildParams* out,
                                             uint32_t* status) {
    float4 r = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (uint32_t b = threadIdx.x; b < nb; b += kBlock) r = minmax4(r, partials[b]);
    if (nb == 0)
        for (uint32_t i = threadIdx.x; i < n; i += kBlock) r = minmax4(r, bounds_item(xs[i], ys[i]));
    r = block_minmax4(r);
    if (threadIdx.x != 0) return;
    if (status) flag_nonfinite(r, status);
    uint64_t mnx64, mny64, mxx64, mxy64;
    if (cb.use) {
        mnx64 = bh_sfp_f64_bits(cb.minx);
        mny64 = bh_sfp_f64_bits(cb.miny);
        mxx64 = bh_sfp_f64_bits(cb.maxx);
        mxy64 = bh_sfp_f64_bits(cb.maxy);
    } else {
        mnx64 = bh_sfp_from_f32(r.x);
        mny64 = bh_sfp_from_f32(r.y);
        mxx64 = bh_sfp_from_f32(r.z);
        mxy64 = bh_sfp_from_f32(r.w);
    }
    fill_params(out, r, mnx64, mny64, mxx64, mxy64, tree_mode, n);
}

__global__ __launch_bounds__(kBlock) void k_bounds_final(const float4* __restrict__ partials,
                                                         uint32_t nb, uint32_t n,
                                                         BuildParams* __restrict__ prm,
                                                         uint32_t tree_mode, CallerBounds cb,
                                                         uint32_t* __restrict__ status) {
    bounds_final(partials, nb, nullptr, nullptr, n, tree_mode, cb, prm, status);
}

// batched systems: bounds per system from per-block partials over each system's blocks
__global__ __launch_bounds__(kBlock) void k_bounds_seg_partial(const float* __restrict__ xs,
                                                               const float* __restrict__ ys,
                                                               const uint2* __restrict__ blk,
                                                               float4* __restrict__ partials) {
    const uint2 bk = blk[blockIdx.x];  // (first particle, count)
    float4 r = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = threadIdx.x; i < bk.y; i += kBlock)
        r = minmax4(r, bounds_item(xs[bk.x + i], ys[bk.x + i]));
    r = block_minmax4(r);
    if (threadIdx.x == 0) partials[blockIdx.x] = r;
}

// one block per system: partials [blk_off[s], blk_off[s+1]) -> sys_prm[s]
__global__ __launch_bounds__(kBlock) void k_bounds_seg_final(const float4* __restrict__ partials,
                                                             const uint32_t* __restrict__ blk_off,
                                                             const uint32_t* __restrict__ sys_off,
                                                             BuildParams* __restrict__ sys_prm,
                                                             BuildParams* __restrict__ prm,
                                                             uint32_t* __restrict__ status) {
    const uint32_t s = blockIdx.x;
    float4 r = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (uint32_t b = blk_off[s] + threadIdx.x; b < blk_off[s + 1]; b += kBlock)
        r = minmax4(r, partials[b]);
    r = block_minmax4(r);
    if (threadIdx.x != 0) return;
    flag_nonfinite(r, status);
    fill_params(sys_prm + s, r, bh_sfp_from_f32(r.x), bh_sfp_from_f32(r.y), bh_sfp_from_f32(r.z),
                bh_sfp_from_f32(r.w), kTreeQuadTree, sys_off[s + 1] - sys_off[s]);
    if (s == 0) {
        prm->n = sys_off[gridDim.x];
        prm->max_level = 0;
        prm->overfull_leaves = 0;
    }
}

__device__ void fill_params(BuildParams* prm, float4 r, uint64_t mnx64, uint64_t mny64,
                            uint64_t mxx64, uint64_t mxy64, uint32_t tree_mode, uint32_t n) {
    uint64_t side;
    if (tree_mode == kTreeQuadTree)
        side = bh_sfp_quadtree_side(mnx64, mny64, mxx64, mxy64);
    else if (tree_mode == kTreeGpuRef)  // createRoot: the larger FP32 extent (.cu:78-94)
        side = bh_sfp_from_f32(fmaxf(r.z - r.x, r.w - r.y));
    else
        side = bh_sfp_morton_extent(mnx64, mny64, mxx64, mxy64);
    if ((side & ~BH_SFP_SIGN) == 0) side = 0x3FF0000000000000ull;  // all points coincide: side 1
    prm->minx = r.x;
    prm->miny = r.y;
    prm->maxx = r.z;
    prm->maxy = r.w;
    prm->minx64 = mnx64;
    prm->miny64 = mny64;
    prm->neg_minx64 = bh_sfp_neg(mnx64);
    prm->neg_miny64 = bh_sfp_neg(mny64);
    prm->side64 = side;
    prm->quant = bh_sfp_quant_prepare(side);
    prm->side = bh_sfp_to_f32(side);
    prm->n = n;
    prm->max_level = 0;
    prm->overfull_leaves = 0;
}

// ------------------------------------------------------------------------------------------
// Morton codes: bit-exact with the reference's FP64 rule via integer emulation
// ------------------------------------------------------------------------------------------
// One particle's state as the gather after the sort reads it: x, y, mass and index in one record,
// a single line of random access where four arrays are four (1M particles in random order, with
// velocities known to be zero: 80 -> 22 us; 4M 467 -> 102; for 2 and 17 us more here).
__device__ __forceinline__ void pack_state(float4* __restrict__ pk, uint32_t i, float x, float y,
                                           const float* __restrict__ m,
                                           const uint32_t* __restrict__ id) {
    pk[i] = make_float4(x, y, m[i], __uint_as_float(id[i]));
}

// Every block derives the root square from the partial bounds itself (block 0 records it): a
// launch of its own for that cost 5 us of every build (70k points: 14 -> 10 us with the codes).
template <typename K, int ITEMS>
__global__ __launch_bounds__(kBlock) void k_morton(const float* __restrict__ xs,
                                                   const float* __restrict__ ys,
                                                   const float* __restrict__ ms,
                                                   const uint32_t* __restrict__ ids, uint32_t n,
                                                   const float4* __restrict__ partials,
                                                   uint32_t nb, uint32_t tree_mode,
                                                   CallerBounds cb, BuildParams* __restrict__ prm,
                                                   uint32_t* __restrict__ status, int B,
                                                   K* __restrict__ keys,
                                                   uint32_t* __restrict__ vals,
                                                   float4* __restrict__ pk) {
    __shared__ BuildParams s_prm;
    const uint32_t base = blockIdx.x * (kBlock * ITEMS) + threadIdx.x;
    float x[ITEMS], y[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = min(base + r * kBlock, n - 1);
        x[r] = xs[i];
        y[r] = ys[i];
    }
    bounds_final(partials, nb, xs, ys, n, tree_mode, cb, &s_prm,
                 blockIdx.x == 0 ? status : nullptr);
    if (threadIdx.x == 0) s_prm.n_nodes = 0;
    __syncthreads();
    static_assert(sizeof(BuildParams) % 4 == 0 && sizeof(BuildParams) / 4 <= kBlock, "one word each");
    if (blockIdx.x == 0 && threadIdx.x < sizeof(BuildParams) / 4)
        reinterpret_cast<uint32_t*>(prm)[threadIdx.x] =
            reinterpret_cast<const uint32_t*>(&s_prm)[threadIdx.x];
    const bh_sfp_quant Q = s_prm.quant;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = base + r * kBlock;
        if (i >= n) return;
        const uint64_t dx = bh_sfp_add(bh_sfp_from_f32(x[r]), s_prm.neg_minx64);
        const uint64_t dy = bh_sfp_add(bh_sfp_from_f32(y[r]), s_prm.neg_miny64);
        const uint64_t qx = bh_sfp_quantize(dx, Q, B);
        const uint64_t qy = bh_sfp_quantize(dy, Q, B);
        K code;
        if (sizeof(K) == 4)
            code = (K)((bh_spread16((uint32_t)qy) << 1) | bh_spread16((uint32_t)qx));
        else
            code = (K)((bh_spread32(qy) << 1) | bh_spread32(qx));
        keys[i] = code;
        vals[i] = i;
        pack_state(pk, i, x[r], y[r], ms, ids);
    }
}

// The tree of the reference's GPU step (NBodySolverGpuBH: createRoot, createChildren,
// nBodySolverGpuBH.cu:78-200): root centred on the bounding box (FP32 midpoint) with side the
// larger FP32 extent; every cell splits at its centre, a point equal to the centre coordinate
// going low; child centres c +- 0.25 l and side 0.5 l in FP32 as there. Each point descends
// `depth` levels by those comparisons; the code holds its path two bits per level, x on the
// even bit as in the Morton codes (the reference's child order A, B, C, D is (x, y) =
// (low, low), (low, high), (high, low), (high, high); only the storage order differs), in the
// top 2 depth bits of the 32-bit key.
__global__ __launch_bounds__(kBlock) void k_morton_gpuref(const float* __restrict__ xs,
                                                          const float* __restrict__ ys,
                                                          const float* __restrict__ ms,
                                                          const uint32_t* __restrict__ ids,
                                                          uint32_t n,
                                                          const BuildParams* __restrict__ prm,
                                                          int depth, uint32_t* __restrict__ keys,
                                                          uint32_t* __restrict__ vals,
                                                          float4* __restrict__ pk) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float mnx = prm->minx, mny = prm->miny, mxx = prm->maxx, mxy = prm->maxy;
    float len = fmaxf(mxx - mnx, mxy - mny);
    float cx = (mnx + mxx) * 0.5f, cy = (mny + mxy) * 0.5f;
    const float x = xs[i], y = ys[i];
    uint32_t code = 0;
    for (int l = 0; l < depth; ++l) {
        const bool xh = !(x <= cx), yh = !(y <= cy);
        code = (code << 2) | ((uint32_t)yh << 1) | (uint32_t)xh;
        const float q = 0.25f * len;
        cx = cx + (xh ? q : -q);
        cy = cy + (yh ? q : -q);
        len = 0.5f * len;
    }
    keys[i] = depth > 0 ? code << (32 - 2 * depth) : 0u;
    vals[i] = i;
    pack_state(pk, i, x, y, ms, ids);
}

// batched systems: key = system << 2B | code, with each system's own root square
// Bound by the search for a particle's system (a chain of log2(nsys) loads) beside 44 bytes of
// memory traffic per particle: 205 -> 151 us for 256 systems of 11.1M particles since a block
// searches once.
__global__ __launch_bounds__(kBlock) void k_morton_seg(const float* __restrict__ xs,
                                                       const float* __restrict__ ys,
                                                       const float* __restrict__ ms,
                                                       const uint32_t* __restrict__ ids, uint32_t n,
                                                       const uint32_t* __restrict__ sys_off,
                                                       uint32_t nsys,
                                                       const BuildParams* __restrict__ sys_prm,
                                                       int B, uint64_t* __restrict__ keys,
                                                       uint32_t* __restrict__ vals,
                                                       float4* __restrict__ pk) {
    const uint32_t b0 = blockIdx.x * kBlock, i = b0 + threadIdx.x;
    if (i >= n) return;
    // largest s with sys_off[s] <= i: found for the block's first particle, then among the systems
    // up to its last one (nearly always the same)
    uint32_t lo = 0, hi = nsys;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sys_off[mid] <= b0) lo = mid; else hi = mid;
    }
    for (uint32_t step = 1; hi < nsys && sys_off[hi] < b0 + kBlock; step *= 2)
        hi = min(hi + step, nsys);
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sys_off[mid] <= i) lo = mid; else hi = mid;
    }
    const BuildParams* prm = sys_prm + lo;
    const bh_sfp_quant Q = prm->quant;
    const float x = xs[i], y = ys[i];
    const uint64_t dx = bh_sfp_add(bh_sfp_from_f32(x), prm->neg_minx64);
    const uint64_t dy = bh_sfp_add(bh_sfp_from_f32(y), prm->neg_miny64);
    const uint64_t qx = bh_sfp_quantize(dx, Q, B);
    const uint64_t qy = bh_sfp_quantize(dy, Q, B);
    keys[i] = ((uint64_t)lo << (2 * B)) | (bh_spread32(qy) << 1) | bh_spread32(qx);
    vals[i] = i;
    pack_state(pk, i, x, y, ms, ids);
}

// ------------------------------------------------------------------------------------------
// device-wide exclusive scan of uint32 (reduce / scan partials / downsweep)
// ------------------------------------------------------------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* total) {
    __shared__ uint32_t wsum[kWavesPerBlock];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(x, o, kWave);
        if (lane >= o) x += t;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t off = 0, tot = 0;
    for (int k = 0; k < kWavesPerBlock; ++k) {
        const uint32_t s = wsum[k];
        if (k < w) off += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

// the same for a block of THREADS threads
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive_scan_t(uint32_t v, uint32_t* total) {
    __shared__ uint32_t wsum[THREADS / kWave];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, kWave);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t off = 0, tot = 0;
    for (int k = 0; k < THREADS / kWave; ++k) {
        const uint32_t s = wsum[k];
        if (k < w) off += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

__global__ __launch_bounds__(kBlock) void k_scan_reduce(const uint32_t* __restrict__ in, uint32_t n,
                                                        uint32_t* __restrict__ partials) {
    const uint32_t base = blockIdx.x * kScanTile;
    uint32_t s = 0;
    for (int r = 0; r < kScanItems; ++r) {
        const uint32_t i = base + r * kBlock + threadIdx.x;
        if (i < n) s += in[i];
    }
    uint32_t tot;
    block_exclusive_scan(s, &tot);
    if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kBlock) void k_scan_partials(uint32_t* __restrict__ partials,
                                                          uint32_t nb, uint32_t* __restrict__ total) {
    const uint32_t per = (nb + kBlock - 1) / kBlock;
    const uint32_t lo = threadIdx.x * per;
    const uint32_t hi = min(lo + per, nb);
    uint32_t s = 0;
    for (uint32_t i = lo; i < hi; ++i) s += partials[i];
    uint32_t tot;
    uint32_t run = block_exclusive_scan(s, &tot);
    for (uint32_t i = lo; i < hi; ++i) {
        const uint32_t v = partials[i];
        partials[i] = run;
        run += v;
    }
    if (threadIdx.x == 0 && total) *total = tot;
}

__global__ __launch_bounds__(kBlock) void k_scan_down(const uint32_t* __restrict__ in,
                                                      uint32_t* __restrict__ out, uint32_t n,
                                                      const uint32_t* __restrict__ partials) {
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int r = 0; r < kScanItems; ++r) {
        v[r] = (base + r < n) ? in[base + r] : 0u;
        s += v[r];
    }
    uint32_t tot;
    uint32_t run = block_exclusive_scan(s, &tot) + partials[blockIdx.x];
#pragma unroll
    for (int r = 0; r < kScanItems; ++r) {
        if (base + r < n) out[base + r] = run;
        run += v[r];
    }
}

// ------------------------------------------------------------------------------------------
// LSD radix sort, 8-bit digits, one launch per pass after one counting launch ("one-sweep"),
// for more than kBucketSortMax keys.
//   k_radix_counts: one block per 4096-key tile; the tile's digit counts for every pass (the
//     multiset of digits of a pass does not depend on the order) and the clearing of the tile's
//     look-back words of every pass.
//   k_radix_totals: per (pass, digit) the total over tiles.
//   k_radix_pass: a block takes the next tile ticket, ranks its keys inside each wave with ballot
//     match masks, publishes the tile's digit counts, and gets the tile's global digit offsets
//     by decoupled look-back over the tiles ticketed before it; it then stages the tile in LDS
//     in digit order so global writes come out as contiguous digit runs. The sort is stable.
// A look-back word holds a 2-bit state (0 not ready, 1 tile count, 2 inclusive prefix) above a
// 30-bit count, so one relaxed device-scope atomic carries both and no fence is needed. A block
// only waits on tiles whose tickets were taken before its own (their blocks are running), so
// every wait ends.
// ------------------------------------------------------------------------------------------
// Tiles of 4096 keys for large sorts, 2048 for sorts of at most kSortSmallMax keys (more blocks
// share a small sort). kSortItems* is the tile in keys per thread of a 256-thread block; the
// kernels take a tile with 4 keys per lane, which measured faster in the radix pass than 8 or 16
// keys per lane on fewer waves.
constexpr int kSortItemsLarge = 16, kSortItemsSmall = 8;
constexpr uint32_t kSortSmallMax = 1u << 18;  // sorts up to this size use the small tiles
__host__ __device__ constexpr int sort_tile(int items) { return kBlock * items; }
constexpr int kSortMaxPasses = 8;
constexpr uint32_t kLbCount = 1u << 30, kLbPrefix = 2u << 30, kLbMask = kLbCount - 1;
constexpr int kLbWindow = 8;  // look-back loads in flight per digit
// the sample-based sorts below
constexpr uint32_t kRankSortMax = 8192, kBucketSortMax = 1u << 21;
static_assert(kSortMaxPasses * 256 >= 2048, "bucket look-back words fit the radix sort's");
constexpr int kBucketMax = 2048, kBucketSamples = 8 * kBucketMax, kBucketItems = 4, kBucketItemsMax = 8;
static_assert(kBlock == 256, "one thread per digit");

// The sum of a digit's counts over the tiles before `tile` (> 0), whose words of the digit stand
// `stride` apart from `status` on: kLbWindow tiles per round with independent loads, nearest
// first; stops at the first inclusive prefix (tile 0 always publishes one), waits at a tile not
// ready.
__device__ __forceinline__ uint32_t look_back(const uint32_t* __restrict__ status, uint32_t stride,
                                              uint32_t tile, uint32_t* __restrict__ err,
                                              uint32_t spin_limit) {
    int j = (int)tile - 1;
    uint32_t excl = 0, spins = 0;
    bool done = false;
    while (!done) {
        uint32_t v[kLbWindow];
#pragma unroll
        for (int k = 0; k < kLbWindow; ++k)
            v[k] = j - k >= 0 ? __hip_atomic_load(status + (size_t)(j - k) * stride,
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                              : kLbPrefix;
        int used = 0;
#pragma unroll
        for (int k = 0; k < kLbWindow; ++k) {
            if (done || used < k) continue;  // stopped earlier in this round
            if ((v[k] & ~kLbMask) == 0u) continue;  // not ready: poll again from here
            excl += v[k] & kLbMask;
            done = (v[k] & kLbPrefix) != 0u;
            used = k + 1;
        }
        j -= used;
        if (!done && used < kLbWindow) {
            // never expected: record it and stop waiting. The tile's prefix is then short of the
            // true one, so this and every later tile still place their keys inside [0, n)
            if (++spins > spin_limit) {
                __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
    return excl;
}

template <typename K, int THREADS, int ITEMS>
__global__ __launch_bounds__(THREADS) void k_radix_counts(const K* __restrict__ keys, uint32_t n,
                                                          int passes, uint32_t ntiles,
                                                          uint32_t* __restrict__ counts,
                                                          uint32_t* __restrict__ status) {
    __shared__ uint32_t h[kSortMaxPasses][256];
    for (int i = threadIdx.x; i < kSortMaxPasses * 256; i += THREADS) (&h[0][0])[i] = 0u;
    for (int i = threadIdx.x; i < passes * 256; i += THREADS)
        status[((size_t)(i >> 8) * ntiles + blockIdx.x) * 256 + (i & 255)] = 0u;
    __syncthreads();
    const uint32_t base = blockIdx.x * (THREADS * ITEMS);
    K k[ITEMS];  // all loads issued before the first use
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = base + r * THREADS + threadIdx.x;
        k[r] = i < n ? keys[i] : (K)0;
    }
    // A wave holds 64 consecutive keys; each run of equal digits among neighbouring lanes is
    // counted by its first lane with one add of the run length. Keys that arrive nearly sorted
    // (particles kept in the previous step's order) would otherwise send most of a wave's adds
    // to one LDS word, which serialises them.
    const int lane = threadIdx.x & 63;
    const uint64_t le = lane_mask_lt() | (1ull << lane);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = base + r * THREADS + threadIdx.x < n;  // invalid lanes are a suffix
        const K prev = (K)__shfl_up((unsigned long long)k[r], 1);
        const uint64_t stops = __ballot(!valid);
        for (int p = 0; p < passes; ++p) {
            const uint32_t d = (uint32_t)(k[r] >> (8 * p)) & 0xFFu;
            const bool head = valid && (lane == 0 || d != ((uint32_t)(prev >> (8 * p)) & 0xFFu));
            const uint64_t after = (__ballot(head) | stops) & ~le;
            const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
            if (head) atomicAdd(&h[p][d], end - (uint32_t)lane);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < passes * 256; i += THREADS)
        counts[(size_t)i * ntiles + blockIdx.x] = h[i >> 8][i & 255];
}

// one wave per (pass, digit) row of counts; block 0 also clears the pass tickets
__global__ __launch_bounds__(kBlock) void k_radix_totals(const uint32_t* __restrict__ counts,
                                                         uint32_t ntiles, int passes,
                                                         uint32_t* __restrict__ totals,
                                                         uint32_t* __restrict__ tickets) {
    if (blockIdx.x == 0 && threadIdx.x < kSortMaxPasses) tickets[threadIdx.x] = 0u;
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (row >= (uint32_t)passes * 256u) return;
    unsigned long long s = 0;
    for (uint32_t j = lane; j < ntiles; j += kWave) s += counts[(size_t)row * ntiles + j];
    s = wave_sum_u64(s);
    if (lane == 0) totals[row] = (uint32_t)s;
}

template <typename K, int THREADS, int ITEMS>
__global__ __launch_bounds__(THREADS) void k_radix_pass(const K* __restrict__ keys_in,
                                                       const uint32_t* __restrict__ vals_in,
                                                       K* __restrict__ keys_out,
                                                       uint32_t* __restrict__ vals_out,
                                                       uint32_t n, int shift,
                                                       const uint32_t* __restrict__ totals,
                                                       uint32_t* __restrict__ status,
                                                       uint32_t* __restrict__ ticket,
                                                       uint32_t* __restrict__ err,
                                                       uint32_t spin_limit) {
    constexpr int kTile = THREADS * ITEMS, kWaveKeys = kWave * ITEMS, kW = THREADS / kWave;
    // After a give-up the keys of the next pass no longer match the digit totals, and placing
    // them could write past the end: every later block leaves at once (the build reports the
    // error and its gather falls back to the identity order).
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
    static_assert(THREADS >= 256, "one thread per digit");
    __shared__ K s_keys[kTile];
    __shared__ uint32_t s_vals[kTile];
    __shared__ uint32_t s_wave[kW][256];  // wave-local counts, then wave offsets
    __shared__ uint32_t s_start[256];                  // tile-local start of each digit
    __shared__ uint32_t s_base[256];                   // global start of each digit for this tile
    __shared__ uint32_t s_tile;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_tile = atomicAdd(ticket, 1u);
    for (int d = threadIdx.x; d < kW * 256; d += THREADS) (&s_wave[0][0])[d] = 0u;
    __syncthreads();
    const uint32_t tile = s_tile;

    const uint32_t wbase = tile * kTile + w * kWaveKeys;
    const uint64_t lt = lane_mask_lt();
    K key[ITEMS];
    uint32_t val[ITEMS];
    uint32_t rank[ITEMS];
    // all loads are issued before the ranking (whose LDS traffic would otherwise make each
    // item wait for its own load)
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = wbase + r * kWave + lane;
        key[r] = i < n ? keys_in[i] : (K)0;
        val[r] = i < n ? vals_in[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = wbase + r * kWave + lane < n;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 0xFFu;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bits = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bits : ~bits;
        }
        const uint32_t before = s_wave[w][d];
        rank[r] = before + (uint32_t)__popcll(peers & lt);
        const bool leader = valid && ((peers & lt) == 0);
        if (leader) s_wave[w][d] = before + (uint32_t)__popcll(peers);
        if (!valid) rank[r] = 0xFFFFFFFFu;
    }
    __syncthreads();
    {
        // threads 0..255 own one digit each; the scans take every thread of the block
        const int d = threadIdx.x & 255;
        const bool dig = threadIdx.x < 256;
        uint32_t cnt = 0;
        if (dig) {
            for (int k = 0; k < kW; ++k) {
                const uint32_t c = s_wave[k][d];
                s_wave[k][d] = cnt;
                cnt += c;
            }
        }
        uint32_t tot;
        const uint32_t start = block_exclusive_scan_t<THREADS>(cnt, &tot);
        if (dig) s_start[d] = start;
        uint32_t* mine = status + (size_t)tile * 256 + d;
        uint32_t excl = 0;
        if (tile == 0) {  // block-uniform: the first tile starts at the digit's global offset
            excl = block_exclusive_scan_t<THREADS>(dig ? totals[d] : 0u, &tot);
        } else if (dig) {
            __hip_atomic_store(mine, kLbCount | cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            excl = look_back(status + d, 256, tile, err, spin_limit);
        }
        if (dig) {
            __hip_atomic_store(mine, kLbPrefix | (excl + cnt), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            s_base[d] = excl;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        if (rank[r] == 0xFFFFFFFFu) continue;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 0xFFu;
        const uint32_t pos = s_start[d] + s_wave[w][d] + rank[r];
        s_keys[pos] = key[r];
        s_vals[pos] = val[r];
    }
    __syncthreads();
    const uint32_t tile_n = min((uint32_t)kTile, n - tile * kTile);
    for (uint32_t p = threadIdx.x; p < tile_n; p += THREADS) {
        const K k = s_keys[p];
        const uint32_t d = (uint32_t)(k >> shift) & 0xFFu;
        const uint32_t g = s_base[d] + (p - s_start[d]);
        keys_out[g] = k;
        vals_out[g] = s_vals[p];
    }
}

// ------------------------------------------------------------------------------------------
// Sorts of up to kBucketSortMax keys. vals holds 0 .. n-1 on entry, so an order by (key, value)
// is the stable order, and every pair is distinct.
//   k_rank_sort: each key's rank is counted against all others, 64 keys per block. The other key
//     is a scalar operand, so a comparison is two vector instructions. One launch; used for whole
//     sorts of at most kRankSortMax keys and for the sample of the larger ones.
//   k_bucket_prepare: a sample of the keys, one from each of equal strata of the input, and the
//     clearing of the look-back words.
//   k_rank_sort on the sample: every bucket's share of it ends at a splitter (key, position).
//   k_bucket_count: each key's bucket by binary search among the splitters in LDS, kept as a
//     16-bit id (equal keys spread over buckets by position); per-tile bucket counts with
//     decoupled look-back over the tiles, as in k_radix_pass.
//   k_bucket_scatter: keys and values to their bucket, staged in LDS so that a tile's keys of one
//     bucket are written as a run. No waits: the look-back words now hold every tile's prefix.
//   k_bucket_sort: one block per bucket merge-sorts its pairs in LDS. A bucket that outgrew LDS (a
//     sample that missed the distribution) is sorted in pieces that its block merges through
//     memory: slow, and right.
// Three passes over the keys and five launches instead of the radix sort's nine and ten (64-bit
// keys), whose waits for earlier tiles are paid once. Measured, radix sort -> this: 2k keys 52 ->
// 8 us (and nine launches fewer), 70k 85 -> 55 beside another kernel, 1M 173 -> 99, 1.5M (batch)
// 217 -> 143; at 4M keys 382 -> 357 (buckets of 2048), within the spread of the passes, so
// larger sorts keep the radix sort: it needs no sample to hold.
// In k_bucket_sort ranking runs of 64 by lane broadcasts before the merges (1M: 57 us instead of
// 46) and merging four runs at a time by binary searches (90 us) were slower.
// ------------------------------------------------------------------------------------------
constexpr int kRankWaves = 16;

template <typename K>
__device__ __forceinline__ bool pair_less(K ka, uint32_t va, K kb, uint32_t vb) {
    return ka < kb || (ka == kb && va < vb);
}

__device__ __forceinline__ uint32_t lane_value(uint32_t x, int j) {
    return (uint32_t)__builtin_amdgcn_readlane((int)x, j);
}
__device__ __forceinline__ uint64_t lane_value(uint64_t x, int j) {
    return ((uint64_t)lane_value((uint32_t)(x >> 32), j) << 32) | lane_value((uint32_t)x, j);
}

// how many of the wave's pairs (qk, qv) stand before (k, v)
template <typename K>
__device__ __forceinline__ uint32_t lanes_before(K qk, uint32_t qv, K k, uint32_t v) {
    uint32_t c = 0;
#pragma unroll 8
    for (int j = 0; j < kWave; ++j)
        c += pair_less(lane_value(qk, j), lane_value(qv, j), k, v) ? 1u : 0u;
    return c;
}


template <typename K, bool SPLIT>
__global__ __launch_bounds__(kRankWaves * kWave) void k_rank_sort(const K* __restrict__ keys,
                                                                  const uint32_t* __restrict__ vals,
                                                                  uint32_t n,
                                                                  uint32_t per,
                                                                  K* __restrict__ keys_out,
                                                                  uint32_t* __restrict__ vals_out) {
    __shared__ uint32_t s_rank[kWave];
    const uint32_t lane = threadIdx.x & 63, b = blockIdx.x, i = b * kWave + lane;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const K k = i < n ? keys[i] : (K)0;
    if (threadIdx.x < kWave) s_rank[lane] = 0u;
    __syncthreads();
    // keys equal to this one count when they stand before it
    const uint32_t chunks = (n + kWave - 1) / kWave;
    uint32_t rank = 0;
    for (uint32_t c = w; c < chunks; c += kRankWaves) {
        const K* __restrict__ q = keys + c * kWave;
        if (c == b || c + 1 == chunks) {
            const uint32_t e = c * kWave + lane;
            rank += lanes_before(e < n ? keys[e] : ~(K)0, e, k, i);
        } else if (c < b) {
#pragma unroll 16
            for (int j = 0; j < kWave; ++j) rank += q[j] <= k ? 1u : 0u;
        } else {
#pragma unroll 16
            for (int j = 0; j < kWave; ++j) rank += q[j] < k ? 1u : 0u;
        }
    }
    atomicAdd(&s_rank[lane], rank);
    __syncthreads();
    if (threadIdx.x >= kWave || i >= n) return;
    rank = s_rank[lane];
    if (SPLIT) {
        if (rank == 0 || (rank & (per - 1))) return;
        rank = rank / per - 1;
    }
    keys_out[rank] = k;
    vals_out[rank] = vals[i];
}

template <typename K>
__global__ __launch_bounds__(kBlock) void k_bucket_prepare(const K* __restrict__ keys, uint32_t n,
                                                           uint32_t samples, K* __restrict__ skey,
                                                           uint32_t* __restrict__ spos,
                                                           uint32_t* __restrict__ status,
                                                           uint32_t words,
                                                           uint32_t* __restrict__ ticket) {
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j == 0) *ticket = 0u;
    for (uint32_t i = j; i < words; i += gridDim.x * kBlock) status[i] = 0u;
    if (j >= samples) return;
    // a scrambled place in the stratum, so that a period in the input is not met in step
    const uint32_t p0 = (uint32_t)((uint64_t)n * j / samples);
    const uint32_t p1 = (uint32_t)((uint64_t)n * (j + 1) / samples);  // > p0: n >= samples
    uint32_t h = j * 0x9E3779B1u;
    h ^= h >> 15;
    h *= 0x85EBCA77u;
    const uint32_t p = p0 + (uint32_t)(((uint64_t)h * (p1 - p0)) >> 32);
    skey[j] = keys[p];
    spos[j] = p;
}

template <typename K, int THREADS>
__global__ __launch_bounds__(THREADS) void k_bucket_count(const K* __restrict__ keys, uint32_t n,
                                                          uint32_t buckets,
                                                          const K* __restrict__ split_key,
                                                          const uint32_t* __restrict__ split_pos,
                                                          uint16_t* __restrict__ id,
                                                          uint32_t* __restrict__ status,
                                                          uint32_t* __restrict__ ticket,
                                                          uint32_t* __restrict__ err,
                                                          uint32_t spin_limit) {
    constexpr int kItems = kBucketItems;
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
    __shared__ K sk[kBucketMax];
    __shared__ uint32_t sp[kBucketMax];
    __shared__ uint32_t hist[kBucketMax];
    __shared__ uint32_t s_tile;
    if (threadIdx.x == 0) s_tile = atomicAdd(ticket, 1u);
    for (uint32_t d = threadIdx.x; d < buckets; d += THREADS) {
        hist[d] = 0u;
        if (d + 1 < buckets) {
            sk[d] = split_key[d];
            sp[d] = split_pos[d];
        }
    }
    __syncthreads();
    const uint32_t tile = s_tile, base = tile * (THREADS * kItems);
    const int lane = threadIdx.x & 63;
    const uint64_t le = lane_mask_lt() | (1ull << lane);
    K k[kItems];
    uint32_t lo[kItems], len = buckets - 1;
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const uint32_t i = base + r * THREADS + threadIdx.x;
        k[r] = i < n ? keys[i] : (K)0;
        lo[r] = 0;
    }
    // splitters below (key, position), for the thread's keys side by side
    while (len) {
        const uint32_t half = (len + 1) >> 1;
#pragma unroll
        for (int r = 0; r < kItems; ++r) {
            const uint32_t i = base + r * THREADS + threadIdx.x;
            const uint32_t mid = lo[r] + half - 1;
            const K s = sk[mid];
            bool below = s < k[r];
            if (s == k[r]) below = sp[mid] < i;
            lo[r] = below ? mid + 1 : lo[r];
        }
        len -= half;
    }
    // runs of equal buckets among neighbouring lanes count with one add (nearly sorted keys)
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const uint32_t i = base + r * THREADS + threadIdx.x;
        const bool valid = i < n;
        const uint32_t prev = __shfl_up(lo[r], 1, kWave);
        const bool head = valid && (lane == 0 || lo[r] != prev);
        const uint64_t after = (__ballot(head) | __ballot(!valid)) & ~le;
        const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
        if (head) atomicAdd(&hist[lo[r]], end - (uint32_t)lane);
        if (valid) id[i] = (uint16_t)lo[r];
    }
    __syncthreads();
    uint32_t* mine = status + (size_t)tile * buckets;
    for (uint32_t d = threadIdx.x; d < buckets; d += THREADS)
        __hip_atomic_store(mine + d, (tile ? kLbCount : kLbPrefix) | hist[d], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    if (tile == 0) return;
    for (uint32_t d = threadIdx.x; d < buckets; d += THREADS) {
        const uint32_t excl = look_back(status + d, buckets, tile, err, spin_limit);
        __hip_atomic_store(mine + d, kLbPrefix | (excl + hist[d]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

// start[d] = sum of count(0 .. d-1)
template <int THREADS, typename F>
__device__ __forceinline__ void bucket_starts(uint32_t buckets, uint32_t* start, F count) {
    constexpr int kPer = kBucketMax / THREADS;
    uint32_t c[kPer], s = 0, tot;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const uint32_t d = threadIdx.x * kPer + q;
        c[q] = d < buckets ? count(d) : 0u;
        s += c[q];
    }
    uint32_t run = block_exclusive_scan_t<THREADS>(s, &tot);
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const uint32_t d = threadIdx.x * kPer + q;
        if (d < buckets) start[d] = run;
        run += c[q];
    }
}

template <typename K, int THREADS>
__global__ __launch_bounds__(THREADS) void k_bucket_scatter(const K* __restrict__ keys,
                                                            const uint32_t* __restrict__ vals,
                                                            uint32_t n, uint32_t buckets,
                                                            const uint16_t* __restrict__ id,
                                                            const uint32_t* __restrict__ status,
                                                            const uint32_t* __restrict__ err,
                                                            K* __restrict__ keys_out,
                                                            uint32_t* __restrict__ vals_out,
                                                            uint32_t* __restrict__ starts) {
    constexpr int kItems = kBucketItems, kTile = THREADS * kItems;
    if (*err != 0u) return;  // the counts are not whole: nothing is placed
    __shared__ K s_key[kTile];
    __shared__ uint32_t s_val[kTile];
    __shared__ uint16_t s_id[kTile];
    __shared__ uint32_t hist[kBucketMax], first[kBucketMax], place[kBucketMax];
    const uint32_t tile = blockIdx.x, base = tile * kTile;
    const int lane = threadIdx.x & 63;
    K k[kItems];
    uint32_t v[kItems], d[kItems], rank[kItems];
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const uint32_t i = base + r * THREADS + threadIdx.x;
        k[r] = i < n ? keys[i] : (K)0;
        v[r] = i < n ? vals[i] : 0u;
        d[r] = i < n ? id[i] : 0u;
    }
    for (uint32_t q = threadIdx.x; q < buckets; q += THREADS) hist[q] = 0u;
    const uint32_t* last = status + (size_t)(gridDim.x - 1) * buckets;
    bucket_starts<THREADS>(buckets, place, [&](uint32_t q) { return last[q] & kLbMask; });
    __syncthreads();
    const uint64_t le = lane_mask_lt() | (1ull << lane);
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const bool valid = base + r * THREADS + threadIdx.x < n;
        const uint32_t prev = __shfl_up(d[r], 1, kWave);
        const bool head = valid && (lane == 0 || d[r] != prev);
        const uint64_t heads = __ballot(head);
        const uint64_t after = (heads | __ballot(!valid)) & ~le;
        const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
        const uint64_t upto = heads & le;
        const int mine = upto ? 63 - (int)__builtin_clzll(upto) : 0;  // the head of my run
        uint32_t at = 0;
        if (head) at = atomicAdd(&hist[d[r]], end - (uint32_t)lane);
        rank[r] = __shfl(at, mine, kWave) + (uint32_t)(lane - mine);
    }
    __syncthreads();
    if (tile == 0)
        for (uint32_t q = threadIdx.x; q < buckets; q += THREADS) starts[q] = place[q];
    else
        for (uint32_t q = threadIdx.x; q < buckets; q += THREADS)
            place[q] += status[(size_t)(tile - 1) * buckets + q] & kLbMask;
    bucket_starts<THREADS>(buckets, first, [&](uint32_t q) { return hist[q]; });
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        if (base + r * THREADS + threadIdx.x >= n) continue;
        const uint32_t p = first[d[r]] + rank[r];
        s_key[p] = k[r];
        s_val[p] = v[r];
        s_id[p] = (uint16_t)d[r];
    }
    __syncthreads();
    const uint32_t cnt = min((uint32_t)kTile, n - base);
    for (uint32_t p = threadIdx.x; p < cnt; p += THREADS) {
        const uint32_t q = s_id[p], g = place[q] + (p - first[q]);
        keys_out[g] = s_key[p];
        vals_out[g] = s_val[p];
    }
}

// Merge sort of the n <= THREADS * ITEMS pairs in sk / sv, in place. The slots from n up to
// THREADS * ITEMS are filled with pairs above every other (no value is 2^32 - 1).
template <typename K, int THREADS, int ITEMS>
__device__ __forceinline__ void block_merge_sort(K* sk, uint32_t* sv, uint32_t n) {
    const uint32_t at = threadIdx.x * ITEMS;
    K k[ITEMS];
    uint32_t v[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        k[i] = at + i < n ? sk[at + i] : ~(K)0;
        v[i] = at + i < n ? sv[at + i] : 0xFFFFFFFFu;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)  // odd-even transposition within the thread
#pragma unroll
        for (int i = r & 1; i + 1 < ITEMS; i += 2) {
            const bool sw = pair_less(k[i + 1], v[i + 1], k[i], v[i]);
            const K ka = sw ? k[i + 1] : k[i], kb = sw ? k[i] : k[i + 1];
            const uint32_t va = sw ? v[i + 1] : v[i], vb = sw ? v[i] : v[i + 1];
            k[i] = ka;
            k[i + 1] = kb;
            v[i] = va;
            v[i + 1] = vb;
        }
    for (uint32_t w = ITEMS; w < n; w <<= 1) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            sk[at + i] = k[i];
            sv[at + i] = v[i];
        }
        __syncthreads();
        const uint32_t a0 = at & ~(2 * w - 1), b0 = a0 + w, diag = at - a0;
        if (b0 >= n) continue;  // the second run is filling alone
        // runs [a0, b0) and [b0, b0 + w): the outputs from `diag` on take the first from a0 + lo
        uint32_t lo = diag > w ? diag - w : 0u, hi = min(diag, w);
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1, o = b0 + diag - 1 - mid;
            const K ka = sk[a0 + mid], kb = sk[o];
            bool less = ka < kb;
            if (ka == kb) less = sv[a0 + mid] < sv[o];
            lo = less ? mid + 1 : lo;
            hi = less ? hi : mid;
        }
        uint32_t ia = a0 + lo, ib = b0 + diag - lo;
        const uint32_t b1 = b0 + w;
        K ka = sk[min(ia, b0 - 1)], kb = sk[min(ib, b1 - 1)];
        uint32_t va = sv[min(ia, b0 - 1)], vb = sv[min(ib, b1 - 1)];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const bool a = ib >= b1 || (ia < b0 && pair_less(ka, va, kb, vb));
            k[i] = a ? ka : kb;
            v[i] = a ? va : vb;
            ia += a ? 1u : 0u;
            ib += a ? 0u : 1u;
            if (i + 1 < ITEMS) {
                const uint32_t next = a ? min(ia, b0 - 1) : min(ib, b1 - 1);
                const K kn = sk[next];
                const uint32_t vn = sv[next];
                ka = a ? kn : ka;
                va = a ? vn : va;
                kb = a ? kb : kn;
                vb = a ? vb : vn;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        sk[at + i] = k[i];
        sv[at + i] = v[i];
    }
    __syncthreads();
}

// merge of the sorted runs [a0, b0) and [b0, b1) from one place to another, by the whole block
template <typename K, int THREADS>
__device__ void block_merge_runs(const K* sk, const uint32_t* sv, K* dk, uint32_t* dv, uint32_t a0,
                                 uint32_t b0, uint32_t b1) {
    const uint32_t na = b0 - a0, nb = b1 - b0, per = (na + nb + THREADS - 1) / THREADS;
    const uint32_t d0 = min(threadIdx.x * per, na + nb), d1 = min(d0 + per, na + nb);
    uint32_t lo = d0 > nb ? d0 - nb : 0u, hi = min(d0, na);
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1, o = b0 + d0 - 1 - mid;
        if (pair_less(sk[a0 + mid], sv[a0 + mid], sk[o], sv[o]))
            lo = mid + 1;
        else
            hi = mid;
    }
    uint32_t ia = a0 + lo, ib = b0 + d0 - lo;
    for (uint32_t d = d0; d < d1; ++d) {
        const bool a = ib >= b1 || (ia < b0 && pair_less(sk[ia], sv[ia], sk[ib], sv[ib]));
        const uint32_t s = a ? ia++ : ib++;
        dk[a0 + d] = sk[s];
        dv[a0 + d] = sv[s];
    }
}

template <typename K, int THREADS>
__global__ __launch_bounds__(THREADS) void k_bucket_sort(K* keys, uint32_t* vals, uint32_t n,
                                                         uint32_t buckets,
                                                         const uint32_t* __restrict__ starts,
                                                         const uint32_t* __restrict__ err,
                                                         K* keys_out, uint32_t* vals_out) {
    constexpr uint32_t kCap = THREADS * kBucketItemsMax;
    if (*err != 0u) return;
    __shared__ K sk[kCap];
    __shared__ uint32_t sv[kCap];
    const uint32_t b = blockIdx.x, start = starts[b];
    const uint32_t cnt = (b + 1 < buckets ? starts[b + 1] : n) - start;
    for (uint32_t c0 = 0; c0 < cnt; c0 += kCap) {  // one piece unless the bucket outgrew LDS
        const uint32_t m = min(cnt - c0, kCap), g = start + c0;
        for (uint32_t i = threadIdx.x; i < m; i += THREADS) {
            sk[i] = keys[g + i];
            sv[i] = vals[g + i];
        }
        __syncthreads();
        if (m <= THREADS) block_merge_sort<K, THREADS, 1>(sk, sv, m);
        else if (m <= 2 * THREADS) block_merge_sort<K, THREADS, 2>(sk, sv, m);
        else if (m <= 4 * THREADS) block_merge_sort<K, THREADS, 4>(sk, sv, m);
        else block_merge_sort<K, THREADS, kBucketItemsMax>(sk, sv, m);
        for (uint32_t i = threadIdx.x; i < m; i += THREADS) {
            keys_out[g + i] = sk[i];
            vals_out[g + i] = sv[i];
        }
        __syncthreads();
    }
    if (cnt <= kCap) return;
    K *from_k = keys_out, *to_k = keys;
    uint32_t *from_v = vals_out, *to_v = vals;
    for (uint32_t w = kCap; w < cnt; w *= 2) {
        __threadfence_block();
        __syncthreads();
        for (uint32_t a0 = 0; a0 < cnt; a0 += 2 * w)
            block_merge_runs<K, THREADS>(from_k, from_v, to_k, to_v, start + a0,
                                         start + min(a0 + w, cnt), start + min(a0 + 2 * w, cnt));
        K* tk = from_k; from_k = to_k; to_k = tk;
        uint32_t* tv = from_v; from_v = to_v; to_v = tv;
    }
    __threadfence_block();
    __syncthreads();
    if (from_k != keys_out)
        for (uint32_t i = threadIdx.x; i < cnt; i += THREADS) {
            keys_out[start + i] = from_k[start + i];
            vals_out[start + i] = from_v[start + i];
        }
}

// ------------------------------------------------------------------------------------------
// the particle state gathered into sorted order; tree: leaf level and node count per particle
// ------------------------------------------------------------------------------------------
// The node count of each tile of kTreeTile particles goes to sums: k_tree_emit_heads takes the
// counts of the tiles before its own from there, so the device-wide scan needs no launch of its
// own (three launches of 2 to 4 us each before). The gather has no launch of its own either: its
// random reads are in flight while the block works on its codes.
// vx, vy: null when the velocities are known to be zero (zeros are then written, not gathered).
constexpr int kTreeTile = 1024;
template <typename K>
__global__ __launch_bounds__(kTreeTile) void k_gather_levels(const uint32_t* __restrict__ perm,
                                                        const float4* __restrict__ pk,
                                                        const float* __restrict__ vx,
                                                        const float* __restrict__ vy,
                                                        float* __restrict__ xo,
                                                        float* __restrict__ yo,
                                                        float* __restrict__ mo,
                                                        float* __restrict__ vxo,
                                                        float* __restrict__ vyo,
                                                        uint32_t* __restrict__ ido,
                                                        float4* __restrict__ pos4,
                                                        K* codes, uint32_t n,
                                                        int B, int R, int cap, int fixed_depth,
                                                        uint8_t* __restrict__ lcp1,
                                                        uint32_t* __restrict__ cnt,
                                                        uint32_t* __restrict__ sums,
                                                        const uint32_t* __restrict__ status) {
    __shared__ K s_code[kTreeTile + 2 * kMaxLeafCap];
    __shared__ int8_t s_w[kTreeTile + kMaxLeafCap];
    const int64_t b0 = (int64_t)blockIdx.x * kTreeTile;
    const int64_t i = b0 + threadIdx.x;
    // a build whose sort gave up or whose input is not finite gets an empty tree: every walk over
    // it ends at once (the call reports the error). A sort that gave up leaves no valid
    // permutation either: the input order is kept, with every code 0 (sorted).
    const bool no_sort = status[0] != 0u, failed = no_sort || status[1] != 0u;
    float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
    float qu = 0.0f, qv = 0.0f;
    if (i < (int64_t)n) {
        const uint32_t j = no_sort ? (uint32_t)i : min(perm[i], n - 1);
        q = pk[j];
        if (vx) qu = vx[j];
        if (vy) qv = vy[j];
    }
    const int adaptive = fixed_depth < 0;
    if (adaptive) {
        const int span = kTreeTile + 2 * cap;
        for (int t = threadIdx.x; t < span; t += kTreeTile) {
            const int64_t j = b0 - cap + t;
            s_code[t] = (j >= 0 && j < (int64_t)n) ? codes[j] : (K)0;
        }
        __syncthreads();
        // w(j) = common level of particles j and j+cap: the window [j, j+cap] shares a cell of
        // that level, so a cell holding i splits while some window through i shares it
        for (int t = threadIdx.x; t < kTreeTile + cap; t += kTreeTile) {
            const int64_t j = b0 - cap + t;
            int8_t wv = -1;
            if (j >= 0 && j + cap < (int64_t)n) wv = (int8_t)lcp_level(s_code[t], s_code[t + cap], B);
            s_w[t] = wv;
        }
        __syncthreads();
    }
    uint32_t c = 0;
    if (i < (int64_t)n) {
        xo[i] = q.x;
        yo[i] = q.y;
        mo[i] = q.z;
        vxo[i] = qu;
        vyo[i] = qv;
        ido[i] = __float_as_uint(q.w);
        pos4[i] = make_float4(q.x, q.y, q.z, 0.0f);
        int leaf;
        if (adaptive) {
            int m = -1;
            for (int t = 0; t <= cap; ++t) m = max(m, (int)s_w[threadIdx.x + t]);
            leaf = max(min(m + 1, B), R);  // more than `cap` in the finest cell: stop at depth B
        } else {
            leaf = fixed_depth;
        }
        // levels below R only separate batched systems: every system's tree starts at level R
        const int lp = max((i == 0) ? -1 : lcp_level(codes[i - 1], codes[i], B), R - 1);
        lcp1[i] = (uint8_t)(lp + 1);
        c = (!failed && leaf > lp) ? (uint32_t)(leaf - lp) : 0u;
        cnt[i] = c;
        if (no_sort) codes[i] = 0;
    }
    uint32_t tot;
    block_exclusive_scan_t<kTreeTile>(c, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// k_tree_emit_nodes is bound by its loads: scattered ones (one line per lane) and, past the L2
// (another XCD wrote the data), chains of them. A node's two searches in the sorted codes run side
// by side, start with kProbes codes at distances 1, 2, 4 .. (most cells are small), narrow what is
// still open in LDS (every block holds one code in `stride`, s_key[t] = codes[t * stride]) and end
// with an 8-ary search; only lanes that need a search load for it. A gallop and a binary search
// in memory took up to 2 log2(n) loads one after another for the topmost cells: 16 -> 10 us at 70k
// points, 17 -> 9.5 at 200k, 25 -> 17 at 1M. Blocks of 256: with 1024 threads the scattered loads
// of a small tree meet on few CUs (17 us at 70k), and 6 probes load more than they save.
constexpr int kTreeKeys = 1024, kTreeThreads = 256, kProbes = 4;

// a search for the first j in [a, b) with codes[j] > key, else b
template <typename K>
struct CodeSearch {
    K key;
    uint32_t a, b;
    __device__ __forceinline__ void see(uint32_t j, K c) {  // codes[j] = c; any order of probes
        if (c > key)
            b = min(b, j);
        else
            a = max(a, j + 1);
    }
    __device__ __forceinline__ void table(const K* s_key, uint32_t keys, uint32_t stride) {
        uint32_t u = 0, v = keys;  // first sample above key
        while (u < v) {
            const uint32_t mid = (u + v) >> 1;
            if (s_key[mid] <= key)
                u = mid + 1;
            else
                v = mid;
        }
        if (u) a = max(a, (u - 1) * stride);
        if (u < keys) b = min(b, u * stride);
    }
    __device__ __forceinline__ uint32_t probe(uint32_t t) const {  // t in 0 .. 6, a < b
        const uint32_t len = b - a;
        return a + (len >> 3) * (t + 1) + (((len & 7) * (t + 1)) >> 3);
    }
};

// nodes of particle i: k = noff[i] + t at level lcp1[i] + t, t < cnt[i]. sums: the node counts of the
// tiles or, scanned, the nodes before each tile
__global__ __launch_bounds__(kTreeTile) void k_tree_emit_heads(uint32_t n,
                                                               const uint8_t* __restrict__ lcp1,
                                                               const uint32_t* __restrict__ cnt,
                                                               const uint32_t* __restrict__ sums,
                                                               int scanned,
                                                               uint32_t* __restrict__ noff,
                                                               BuildParams* __restrict__ prm,
                                                               Node* __restrict__ nodes,
                                                               uint4* __restrict__ child4,
                                                               uint32_t cap_nodes) {
    const uint32_t i = blockIdx.x * kTreeTile + threadIdx.x;
    const uint32_t c = i < n ? cnt[i] : 0u;
    const uint32_t l0 = i < n ? lcp1[i] : 0u;
    uint32_t before = 0, all, tot;
    if (scanned) {
        all = sums[blockIdx.x];
    } else {
        for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kTreeTile) before += sums[b];
        block_exclusive_scan_t<kTreeTile>(before, &all);
    }
    const uint32_t base = all + block_exclusive_scan_t<kTreeTile>(c, &tot);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) prm->n_nodes = all + tot;
    if (i >= n) return;
    noff[i] = base;
    for (uint32_t t = 0; t < c; ++t) {
        const uint32_t k = base + t;
        if (k >= cap_nodes) break;  // cannot happen for the capacity the context allocates
        nodes[k].first = i;
        nodes[k].meta = (l0 + t) | (t == 0 ? kMetaHead : 0u) | (t + 1 == c ? kMetaLeaf : 0u);
        child4[k] = make_uint4(kNone, kNone, kNone, kNone);
    }
}

// one thread per node: subtree extent, flags, side and the parent's child slot
template <typename K>
__global__ __launch_bounds__(kTreeThreads) void k_tree_emit_nodes(const K* __restrict__ codes,
                                                            uint32_t n, int B, int R,
                                                            const uint8_t* __restrict__ lcp1,
                                                            const uint32_t* __restrict__ noff,
                                                            const BuildParams* __restrict__ prm,
                                                            const BuildParams* __restrict__ sys_prm,
                                                            int single_child_pp,
                                                            Node* __restrict__ nodes,
                                                            uint32_t* __restrict__ child4,
                                                            uint32_t cap_nodes) {
    __shared__ K s_key[kTreeKeys];
    const uint32_t k = blockIdx.x * kTreeThreads + threadIdx.x;
    const Node n0 = nodes[min(k, cap_nodes - 1)];  // not yet written past the last node
    const uint32_t total = prm->n_nodes;
    if (blockIdx.x * kTreeThreads >= min(total, cap_nodes)) return;
    const uint32_t stride = (n + kTreeKeys - 1) / kTreeKeys, keys = (n + stride - 1) / stride;
    for (uint32_t t = threadIdx.x; t < keys; t += kTreeThreads) s_key[t] = codes[t * stride];
    __syncthreads();
    if (k >= total || k >= cap_nodes) return;
    const uint32_t i = n0.first;
    uint32_t meta = n0.meta;
    const int l = (int)(meta & kMetaLevelMask);
    const K ci = codes[i];
    // end of the cell: first code above its last one (the single root of a one-system tree, level
    // 0, ends at n); first particle of the parent's cell, for the head of a run of nodes
    const bool up = l > 0, back = l > max(R, 1) && (meta & kMetaHead);
    CodeSearch<K> e{(K)0, n, n}, ip{(K)0, 0, 0};
    if (up) e = CodeSearch<K>{ci | (K)(((K)1 << (2 * (B - l))) - 1), i + 1, n};
    if (back) {
        const K lk = ci & ~(K)(((K)1 << (2 * (B - l + 1))) - 1);
        if (lk) ip = CodeSearch<K>{lk - 1, 0, i};
    }
    {
        K q[kProbes], r[kProbes];
        if (up) {
#pragma unroll
            for (uint32_t t = 0; t < kProbes; ++t) q[t] = codes[min(i + (1u << t), n - 1)];
        }
        if (back) {
#pragma unroll
            for (uint32_t t = 0; t < kProbes; ++t) r[t] = codes[i >= (1u << t) ? i - (1u << t) : 0u];
        }
#pragma unroll
        for (uint32_t t = 0; t < kProbes; ++t) {
            if (up && i + (1u << t) < n) e.see(i + (1u << t), q[t]);
            if (ip.b && i >= (1u << t)) ip.see(i - (1u << t), r[t]);
        }
    }
    if (e.b - e.a > (1u << kProbes)) e.table(s_key, keys, stride);
    if (ip.b - ip.a > (1u << kProbes)) ip.table(s_key, keys, stride);
    for (;;) {
        const bool se = e.a < e.b, si = ip.a < ip.b;
        if (!se && !si) break;
        uint32_t je[7], ji[7];
        K q[7], r[7];
#pragma unroll
        for (uint32_t t = 0; t < 7; ++t) {
            je[t] = e.probe(t);
            ji[t] = ip.probe(t);
        }
        if (se) {
#pragma unroll
            for (uint32_t t = 0; t < 7; ++t) q[t] = codes[je[t]];
        }
        if (si) {
#pragma unroll
            for (uint32_t t = 0; t < 7; ++t) r[t] = codes[ji[t]];
        }
#pragma unroll
        for (uint32_t t = 0; t < 7; ++t) {
            if (se) e.see(je[t], q[t]);
            if (si) ip.see(ji[t], r[t]);
        }
    }
    const uint32_t end = e.a;
    const K last = codes[end - 1];
    const uint32_t skip = end < n ? noff[end] : total;
    const uint32_t pk = back ? noff[ip.a] + (uint32_t)(l - 1 - (int)lcp1[ip.a]) : 0u;
    if (meta & kMetaLeaf) {
        meta |= kMetaPP;
    } else if (single_child_pp) {
        const int shc = 2 * (B - l - 1);
        if (((uint32_t)(ci >> shc) & 3u) == ((uint32_t)(last >> shc) & 3u)) meta |= kMetaPP;
    }
    const BuildParams* sp = R ? sys_prm + (uint32_t)(ci >> (2 * (B - R))) : prm;
    const float sl = ldexpf(sp->side, -(l - R));
    Node* nd = nodes + k;
    nd->l2 = sl * sl;
    nd->skip = skip;
    nd->count = end - i;
    nd->meta = meta;
    if (l > R) {
        const uint32_t par = !(meta & kMetaHead) ? k - 1 : pk;
        child4[4ull * par + ((uint32_t)(ci >> (2 * (B - l))) & 3u)] = k;
    }
}

// ------------------------------------------------------------------------------------------
// upward pass: mass, centre of mass and (optionally) second moments
//
// Pass 1: each block owns a chunk of kUpChunk consecutive nodes and settles them level by
// level (deepest first) in LDS; a node whose subtree runs past the chunk end is left for pass
// 2. Those nodes are ancestors of the chunk's end, so there are at most kMaxLevels + 1 of them
// per chunk. Pass 2: one block settles all of them level by level.
// Children are combined in digit order, so the result does not depend on scheduling.
// ------------------------------------------------------------------------------------------
struct Moments {
    float m, x, y, xx, xy, yy;
};

__device__ __forceinline__ Moments leaf_moments(const float4* __restrict__ pos4, uint32_t f,
                                                uint32_t c, bool with_m2) {
    const float4 p0 = pos4[f];
    float M = 0.f, sx = 0.f, sy = 0.f;
    // kLeafBatch loads in flight at a time (pos4 is padded past n; the tail is masked), summed
    // in particle order
    constexpr uint32_t kLeafBatch = 8;
    for (uint32_t j0 = f; j0 < f + c; j0 += kLeafBatch) {
        float4 q[kLeafBatch];
#pragma unroll
        for (uint32_t u = 0; u < kLeafBatch; ++u) q[u] = pos4[min(j0 + u, f + c - 1)];
#pragma unroll
        for (uint32_t u = 0; u < kLeafBatch; ++u) {
            if (j0 + u >= f + c) break;
            M += q[u].z;
            sx = fmaf(q[u].z, q[u].x - p0.x, sx);
            sy = fmaf(q[u].z, q[u].y - p0.y, sy);
        }
    }
    const float inv = (M != 0.f) ? 1.0f / M : 0.f;
    Moments r{M, p0.x + sx * inv, p0.y + sy * inv, 0.f, 0.f, 0.f};
    if (with_m2) {
        for (uint32_t j = f; j < f + c; ++j) {
            const float4 p = pos4[j];
            const float rx = p.x - r.x, ry = p.y - r.y;
            r.xx = fmaf(p.z * rx, rx, r.xx);
            r.xy = fmaf(p.z * rx, ry, r.xy);
            r.yy = fmaf(p.z * ry, ry, r.yy);
        }
    }
    return r;
}

// Fixed-depth trees can hold thousands of points in one leaf (a tight cluster): such leaves
// (more than kBigLeaf points) get their mass and centre of mass from one wave each before the
// chunked pass, which then takes them from the node record.
constexpr uint32_t kBigLeaf = 64;

__global__ __launch_bounds__(kBlock) void k_big_leaf_moments(const float4* __restrict__ pos4,
                                                             Node* __restrict__ nodes,
                                                             const BuildParams* __restrict__ prm,
                                                             uint32_t cap_nodes) {
    const int lane = threadIdx.x & 63;
    const uint32_t k = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (k >= cap_nodes || k >= prm->n_nodes) return;
    const uint32_t meta = nodes[k].meta, f = nodes[k].first, c = nodes[k].count;
    if (!(meta & kMetaLeaf) || c <= kBigLeaf) return;
    const float4 p0 = pos4[f];
    float M = 0.f, sx = 0.f, sy = 0.f;
    for (uint32_t j = f + lane; j < f + c; j += kWave) {
        const float4 q = pos4[j];
        M += q.z;
        sx = fmaf(q.z, q.x - p0.x, sx);
        sy = fmaf(q.z, q.y - p0.y, sy);
    }
    M = wave_sum_f(M);
    sx = wave_sum_f(sx);
    sy = wave_sum_f(sy);
    if (lane == 0) {
        const float inv = (M != 0.f) ? 1.0f / M : 0.f;
        nodes[k].cx = p0.x + sx * inv;
        nodes[k].cy = p0.y + sy * inv;
        nodes[k].mass = M;
    }
}

// combine up to four children (absent ones have m = 0 and are flagged by has[t] = false)
__device__ __forceinline__ Moments combine(const Moments* ch, const bool* has, bool with_m2) {
    // origin: the first child present (selected with constant indices: no private memory)
    float ox = ch[3].x, oy = ch[3].y;
#pragma unroll
    for (int t = 2; t >= 0; --t) {
        if (has[t]) {
            ox = ch[t].x;
            oy = ch[t].y;
        }
    }
    float M = 0.f, px = 0.f, py = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (!has[t]) continue;
        M += ch[t].m;
        px = fmaf(ch[t].m, ch[t].x - ox, px);
        py = fmaf(ch[t].m, ch[t].y - oy, py);
    }
    const float inv = (M != 0.f) ? 1.0f / M : 0.f;
    Moments r{M, ox + px * inv, oy + py * inv, 0.f, 0.f, 0.f};
    if (with_m2) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (!has[t]) continue;
            const float rx = ch[t].x - r.x, ry = ch[t].y - r.y;
            r.xx += ch[t].xx + ch[t].m * rx * rx;
            r.xy += ch[t].xy + ch[t].m * rx * ry;
            r.yy += ch[t].yy + ch[t].m * ry * ry;
        }
    }
    return r;
}

// A block's time is a chain of latencies: node records, then leaf points, then one LDS round per
// level. The child slots are therefore loaded with the records, the level loop covers the chunk's
// own levels only, and small trees take small chunks (rule at launch_upward): 25 -> 12 us at 70k
// points beside another kernel, 27 -> 13 us at 200k, 28 -> 26 us at 1M (60 MB of records).
template <int CHUNK, int THREADS, bool M2>
__global__ __launch_bounds__(THREADS) void k_up_chunk(const float4* __restrict__ pos4,
                                                     Node* __restrict__ nodes,
                                                     const uint4* __restrict__ child4,
                                                     float4* __restrict__ m2,
                                                     const BuildParams* __restrict__ prm,
                                                     uint32_t* __restrict__ deferred,
                                                     uint32_t cap_nodes, int big_done) {
    __shared__ float s_m[CHUNK], s_x[CHUNK], s_y[CHUNK];
    __shared__ float s_xx[M2 ? CHUNK : 1], s_xy[M2 ? CHUNK : 1], s_yy[M2 ? CHUNK : 1];
    __shared__ uint32_t s_maxl, s_minl;
    __shared__ uint32_t s_ndef;
    constexpr int kPer = CHUNK / THREADS;
    const uint32_t total = min(prm->n_nodes, cap_nodes);
    const uint32_t c0 = blockIdx.x * CHUNK;
    uint32_t* my_def = deferred + (size_t)blockIdx.x * kDeferStride;
    if (c0 >= total) {
        if (threadIdx.x == 0) my_def[0] = 0;
        return;
    }
    const uint32_t c1 = min(c0 + CHUNK, total);
    if (threadIdx.x == 0) {
        s_maxl = 0;
        s_minl = 255;
        s_ndef = 0;
    }
    __syncthreads();
    Node nd[kPer];
    uint4 kids[kPer];
    uint32_t lmax = 0, lmin = 255;
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const uint32_t k = c0 + threadIdx.x + r * THREADS;
        if (k < c1) {
            nd[r] = nodes[k];
            kids[r] = child4[k];
            lmax = max(lmax, nd[r].meta & kMetaLevelMask);
            lmin = min(lmin, nd[r].meta & kMetaLevelMask);
        }
    }
    atomicMax(&s_maxl, lmax);
    atomicMin(&s_minl, lmin);
    // leaves first, all at once: their particle loads overlap instead of waiting level by level
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const uint32_t k = c0 + threadIdx.x + r * THREADS;
        if (k >= c1 || !(nd[r].meta & kMetaLeaf)) continue;
        const uint32_t s = k - c0;
        // leaves of more than kBigLeaf points hold their moments already when k_big_leaf_moments
        // ran (fixed-depth trees); otherwise (coincident points at the depth limit of an
        // adaptive tree, rare) this thread sums them
        const Moments mo = (big_done && nd[r].count > kBigLeaf)
                               ? Moments{nd[r].mass, nd[r].cx, nd[r].cy, 0.f, 0.f, 0.f}
                               : leaf_moments(pos4, nd[r].first, nd[r].count, M2);
        s_m[s] = mo.m; s_x[s] = mo.x; s_y[s] = mo.y;
        if (M2) { s_xx[s] = mo.xx; s_xy[s] = mo.xy; s_yy[s] = mo.yy; }
    }
    __syncthreads();
    for (int L = (int)s_maxl; L >= (int)s_minl; --L) {
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
            const uint32_t k = c0 + threadIdx.x + r * THREADS;
            if (k >= c1 || (int)(nd[r].meta & kMetaLevelMask) != L) continue;
            const uint32_t s = k - c0;
            if (nd[r].meta & kMetaLeaf) {
                continue;
            } else if (nd[r].skip <= c1) {
                const uint32_t ci[4] = {kids[r].x, kids[r].y, kids[r].z, kids[r].w};
                Moments ch[4];
                bool has[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    has[t] = ci[t] != kNone;
                    const uint32_t q = has[t] ? ci[t] - c0 : s;
                    ch[t] = Moments{s_m[q], s_x[q], s_y[q], M2 ? s_xx[q] : 0.f,
                                    M2 ? s_xy[q] : 0.f, M2 ? s_yy[q] : 0.f};
                }
                const Moments mo = combine(ch, has, M2);
                s_m[s] = mo.m; s_x[s] = mo.x; s_y[s] = mo.y;
                if (M2) { s_xx[s] = mo.xx; s_xy[s] = mo.xy; s_yy[s] = mo.yy; }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const uint32_t k = c0 + threadIdx.x + r * THREADS;
        if (k >= c1) continue;
        const uint32_t s = k - c0;
        if ((nd[r].meta & kMetaLeaf) || nd[r].skip <= c1) {
            nodes[k].cx = s_x[s];
            nodes[k].cy = s_y[s];
            nodes[k].mass = s_m[s];
            if (M2) m2[k] = make_float4(s_xx[s], s_xy[s], s_yy[s], 0.f);
        } else {
            // ancestors of the chunk end (at most one per level)
            const uint32_t slot = atomicAdd(&s_ndef, 1u);
            if (slot < kDeferStride - 1) my_def[1 + slot] = k;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) my_def[0] = min(s_ndef, (uint32_t)(kDeferStride - 1));
}

__device__ __forceinline__ Moments load_moments(const Node* __restrict__ nodes,
                                                const float4* __restrict__ m2, uint32_t q,
                                                bool with_m2) {
    Moments r;
    r.m = __hip_atomic_load(&nodes[q].mass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    r.x = __hip_atomic_load(&nodes[q].cx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    r.y = __hip_atomic_load(&nodes[q].cy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    r.xx = r.xy = r.yy = 0.f;
    if (with_m2) {
        r.xx = __hip_atomic_load(&m2[q].x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        r.xy = __hip_atomic_load(&m2[q].y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        r.yy = __hip_atomic_load(&m2[q].z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return r;
}

// Single block of kUpThreads: the nodes left over by k_up_chunk (ancestors of chunk ends),
// deepest level first. With at most kTopMax of them, everything stays on chip: the list is
// compacted into LDS, an LDS hash maps node index -> list entry, the moments of children that
// k_up_chunk settled are loaded once into registers (thread e % kUpThreads owns entry e), and
// the moments of deferred children are passed through LDS from one level to the next. Larger
// lists take the same steps through global memory. Children are combined in digit order
// either way, so the result does not depend on which nodes were deferred.
constexpr int kTopHash = 4096;                                 // hash slots, > kTopMax
constexpr int kTopPer = (kTopMax + kUpThreads - 1) / kUpThreads;  // entries per thread
static_assert(kTopHash >= kTopMax && (kTopHash & (kTopHash - 1)) == 0, "hash size");
static_assert(kTopMax < 65536, "entry indices are 16-bit");

__device__ __forceinline__ uint32_t top_hash(uint32_t k) { return (k * 0x9E3779B1u) >> 20; }

template <bool M2>
__global__ __launch_bounds__(kUpThreads) void k_up_top(Node* __restrict__ nodes,
                                                       const uint4* __restrict__ child4,
                                                       float4* __restrict__ m2,
                                                       const BuildParams* __restrict__ prm,
                                                       const uint32_t* __restrict__ deferred,
                                                       uint32_t* __restrict__ bylevel,
                                                       uint32_t nchunks, uint32_t chunk,
                                                       uint32_t cap_nodes) {
    __shared__ uint32_t s_k[kTopMax];
    __shared__ uint8_t s_l[kTopMax];
    __shared__ uint32_t s_hk[kTopHash];  // node index + 1, 0 = empty
    __shared__ uint16_t s_hv[kTopHash];  // its entry
    __shared__ float s_mo[M2 ? 6 : 3][kTopMax];   // moments of settled entries
    __shared__ uint32_t s_count, s_maxl;
    const uint32_t tid = threadIdx.x;
    const uint32_t total = min(prm->n_nodes, cap_nodes);
    const uint32_t nch = min(nchunks, (total + chunk - 1) / chunk);
    if (tid == 0) {
        s_count = 0;
        s_maxl = 0;
    }
    for (uint32_t i = tid; i < kTopHash; i += kUpThreads) s_hk[i] = 0u;
    __syncthreads();
    // compaction: chunk lists in chunk order
    for (uint32_t b0 = 0; b0 < nch; b0 += kUpThreads) {
        const uint32_t b = b0 + tid;
        const uint32_t c = (b < nch) ? deferred[(size_t)b * kDeferStride] : 0u;
        uint32_t tot;
        const uint32_t off = block_exclusive_scan_t<kUpThreads>(c, &tot);
        const uint32_t base = s_count;
        const uint32_t* lst = deferred + (size_t)b * kDeferStride + 1;
        for (uint32_t j0 = 0; j0 < c; j0 += 8) {  // eight loads in flight
            uint32_t q[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) q[u] = lst[min(j0 + u, c - 1)];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u)
                if (j0 + u < c && base + off + j0 + u < kTopMax) s_k[base + off + j0 + u] = q[u];
        }
        __syncthreads();
        if (tid == 0) s_count = base + tot;
        __syncthreads();
    }
    const uint32_t D = s_count;
    if (D > kTopMax) {
        // large list (many trees: batched systems): the entries bucketed by level with a
        // counting sort into `bylevel`, then each level's bucket settled, deepest first, through
        // global memory. Each node combines its settled children in digit order, so the order
        // inside a bucket does not change any result.
        __shared__ uint32_t s_lc[256], s_lo[256];  // per level: entries, then bucket start
        for (uint32_t i = tid; i < 256; i += kUpThreads) s_lc[i] = 0u;
        __syncthreads();
        const uint32_t entries = nch * (kDeferStride - 1);
        for (uint32_t e = tid; e < entries; e += kUpThreads) {
            const uint32_t b = e / (kDeferStride - 1), slot = e % (kDeferStride - 1);
            const uint32_t* lst = deferred + (size_t)b * kDeferStride;
            if (slot < lst[0]) atomicAdd(&s_lc[nodes[lst[1 + slot]].meta & kMetaLevelMask], 1u);
        }
        __syncthreads();
        if (tid == 0) {
            uint32_t at = 0;
            for (int l = 0; l < 256; ++l) {
                s_lo[l] = at;
                at += s_lc[l];
                s_lc[l] = 0u;
            }
        }
        __syncthreads();
        for (uint32_t e = tid; e < entries; e += kUpThreads) {
            const uint32_t b = e / (kDeferStride - 1), slot = e % (kDeferStride - 1);
            const uint32_t* lst = deferred + (size_t)b * kDeferStride;
            if (slot >= lst[0]) continue;
            const uint32_t k = lst[1 + slot];
            const uint32_t l = nodes[k].meta & kMetaLevelMask;
            bylevel[s_lo[l] + atomicAdd(&s_lc[l], 1u)] = k;
        }
        __syncthreads();
        for (int L = 255; L >= 0; --L) {
            const uint32_t lo = s_lo[L], cnt = s_lc[L];  // the same in every thread
            if (cnt == 0u) continue;
            for (uint32_t i = tid; i < cnt; i += kUpThreads) {
                const uint32_t k = bylevel[lo + i];
                const uint4 cs = child4[k];
                const uint32_t ci[4] = {cs.x, cs.y, cs.z, cs.w};
                Moments ch[4];
                bool has[4];
#pragma unroll
                for (int t2 = 0; t2 < 4; ++t2) {
                    has[t2] = ci[t2] != kNone;
                    ch[t2] = load_moments(nodes, m2, has[t2] ? ci[t2] : k, M2);
                }
                const Moments mo = combine(ch, has, M2);
                __hip_atomic_store(&nodes[k].cx, mo.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_store(&nodes[k].cy, mo.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_store(&nodes[k].mass, mo.m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (M2) {
                    __hip_atomic_store(&m2[k].x, mo.xx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_store(&m2[k].y, mo.xy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_store(&m2[k].z, mo.yy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
            __syncthreads();
        }
        return;
    }
    // on chip: levels and the hash of this thread's entries
    uint32_t lmax = 0;
    uint32_t kk[kTopPer], lev[kTopPer];
    uint4 kids[kTopPer];
#pragma unroll
    for (int r = 0; r < kTopPer; ++r) {
        const uint32_t e = tid + r * kUpThreads;
        kk[r] = e < D ? s_k[e] : 0u;
        lev[r] = e < D ? nodes[kk[r]].meta & kMetaLevelMask : 0u;
        kids[r] = e < D ? child4[kk[r]] : make_uint4(kNone, kNone, kNone, kNone);
    }
#pragma unroll
    for (int r = 0; r < kTopPer; ++r) {
        const uint32_t e = tid + r * kUpThreads;
        if (e >= D) continue;
        const uint32_t l = lev[r];
        s_l[e] = (uint8_t)l;
        lmax = max(lmax, l);
        uint32_t h = top_hash(kk[r]) & (kTopHash - 1);
        while (atomicCAS(&s_hk[h], 0u, kk[r] + 1u) != 0u) h = (h + 1) & (kTopHash - 1);
        s_hv[h] = (uint16_t)e;
    }
    atomicMax(&s_maxl, lmax);
    __syncthreads();
    // children: deferred ones by entry, settled ones loaded once
    Moments ch[kTopPer][4];
    int ce[kTopPer][4];
    bool has[kTopPer][4];
#pragma unroll
    for (int r = 0; r < kTopPer; ++r) {
        const uint32_t ci[4] = {kids[r].x, kids[r].y, kids[r].z, kids[r].w};
#pragma unroll
        for (int t2 = 0; t2 < 4; ++t2) {
            has[r][t2] = ci[t2] != kNone;
            ce[r][t2] = -1;
            ch[r][t2] = Moments{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (!has[r][t2]) continue;
            uint32_t h = top_hash(ci[t2]) & (kTopHash - 1);
            uint32_t key;
            while ((key = s_hk[h]) != 0u && key != ci[t2] + 1u) h = (h + 1) & (kTopHash - 1);
            if (key != 0u) {
                ce[r][t2] = s_hv[h];
            } else {
                const Node q = nodes[ci[t2]];
                ch[r][t2].m = q.mass;
                ch[r][t2].x = q.cx;
                ch[r][t2].y = q.cy;
                if (M2) {
                    const float4 q2 = m2[ci[t2]];
                    ch[r][t2].xx = q2.x;
                    ch[r][t2].xy = q2.y;
                    ch[r][t2].yy = q2.z;
                }
            }
        }
    }
    for (int L = (int)s_maxl; L >= 0; --L) {
#pragma unroll
        for (int r = 0; r < kTopPer; ++r) {
            const uint32_t e = tid + r * kUpThreads;
            if (e >= D || (int)s_l[e] != L) continue;
#pragma unroll
            for (int t2 = 0; t2 < 4; ++t2) {
                const int q = ce[r][t2];
                if (q < 0) continue;
                ch[r][t2] = Moments{s_mo[0][q], s_mo[1][q], s_mo[2][q], M2 ? s_mo[M2 ? 3 : 0][q] : 0.f,
                                    M2 ? s_mo[M2 ? 4 : 0][q] : 0.f, M2 ? s_mo[M2 ? 5 : 0][q] : 0.f};
            }
            const Moments mo = combine(ch[r], has[r], M2);
            s_mo[0][e] = mo.m; s_mo[1][e] = mo.x; s_mo[2][e] = mo.y;
            if (M2) { s_mo[M2 ? 3 : 0][e] = mo.xx; s_mo[M2 ? 4 : 0][e] = mo.xy; s_mo[M2 ? 5 : 0][e] = mo.yy; }
            nodes[kk[r]].cx = mo.x;
            nodes[kk[r]].cy = mo.y;
            nodes[kk[r]].mass = mo.m;
            if (M2) m2[kk[r]] = make_float4(mo.xx, mo.xy, mo.yy, 0.f);
        }
        __syncthreads();
    }
}

// batched systems: the root of system s is the first node of its first particle
__global__ __launch_bounds__(kBlock) void k_batch_roots(const uint32_t* __restrict__ sys_off,
                                                        uint32_t nsys,
                                                        const uint32_t* __restrict__ noff,
                                                        const BuildParams* __restrict__ prm,
                                                        uint32_t* __restrict__ roots) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= nsys) return;
    const uint32_t r = sys_off[s] < sys_off[s + 1] ? noff[sys_off[s]] : kNone;
    roots[s] = r < prm->n_nodes ? r : kNone;  // an empty tree (failed build) has no roots
}

// tree statistics on request: deepest leaf level and leaves at the depth limit holding more
// than the leaf capacity (one partial per block, summed by the host)
__global__ __launch_bounds__(kBlock) void k_tree_stats(const Node* __restrict__ nodes,
                                                       const BuildParams* __restrict__ prm,
                                                       uint32_t cap_nodes, int depth_limit,
                                                       uint32_t leaf_cap,
                                                       uint2* __restrict__ out) {
    uint32_t mx = 0, over = 0;
    const uint32_t total = min(prm->n_nodes, cap_nodes);
    for (uint32_t k = blockIdx.x * kBlock + threadIdx.x; k < total; k += gridDim.x * kBlock) {
        const uint32_t meta = nodes[k].meta;
        if (!(meta & kMetaLeaf)) continue;
        const uint32_t l = meta & kMetaLevelMask;
        mx = max(mx, l);
        if ((int)l == depth_limit && nodes[k].count > leaf_cap) ++over;
    }
    for (int o = 32; o > 0; o >>= 1) {
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, kWave));
        over += (uint32_t)__shfl_xor((int)over, o, kWave);
    }
    __shared__ uint2 red[kWavesPerBlock];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_uint2(mx, over);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint2 r = red[0];
        for (int w = 1; w < kWavesPerBlock; ++w) {
            r.x = max(r.x, red[w].x);
            r.y += red[w].y;
        }
        out[blockIdx.x] = r;
    }
}

// ------------------------------------------------------------------------------------------
// reference slot layout of the fixed-depth Morton tree (nBodySolverFMM_SYM_MORTON.h:117-151,
// 328-470): slot = levelIndex[l] + cell index, firstChildIndex = levelIndex[l+1] + 4 cell
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = v;
}

// the three slot arrays cleared in one launch
__global__ __launch_bounds__(kBlock) void k_clear_slots(uint32_t* __restrict__ a,
                                                        uint32_t* __restrict__ b,
                                                        uint32_t* __restrict__ c, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        a[i] = 0u;
        b[i] = 0u;
        c[i] = 0u;
    }
}

// what a caller did not give: index order, unit masses (m not null), zero velocities (vx not null)
__global__ __launch_bounds__(kBlock) void k_init_state(uint32_t n, uint32_t* __restrict__ id,
                                                       float* __restrict__ m,
                                                       float* __restrict__ vx,
                                                       float* __restrict__ vy) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    id[i] = i;
    if (m) m[i] = 1.0f;
    if (vx) {
        vx[i] = 0.0f;
        vy[i] = 0.0f;
    }
}

__global__ __launch_bounds__(kBlock) void k_tree_slots(const uint32_t* __restrict__ codes,
                                                       const Node* __restrict__ nodes,
                                                       const BuildParams* __restrict__ prm,
                                                       uint32_t cap_nodes, int depth,
                                                       uint32_t* __restrict__ first_child,
                                                       uint32_t* __restrict__ first_particle,
                                                       uint32_t* __restrict__ count) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= cap_nodes || k >= prm->n_nodes) return;
    const Node nd = nodes[k];
    const int l = (int)(nd.meta & kMetaLevelMask);
    const uint32_t cell = (l == 0) ? 0u : (codes[nd.first] >> (2 * (16 - l)));
    const uint32_t li = (uint32_t)((((uint64_t)1 << (2 * l)) - 1) / 3);
    const uint32_t slot = li + cell;
    first_particle[slot] = nd.first;
    count[slot] = nd.count;
    first_child[slot] = (l < depth) ? (uint32_t)((((uint64_t)1 << (2 * (l + 1))) - 1) / 3) + 4u * cell : 0u;
}

// ------------------------------------------------------------------------------------------
// host launchers
// ------------------------------------------------------------------------------------------
static inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

uint32_t bounds_grid(uint32_t n) {
    uint32_t g = div_up(n, kBlock * 8);
    if (g < 1) g = 1;
    if (g > kMaxBoundsBlocks) g = kMaxBoundsBlocks;
    return g;
}

static CallerBounds caller_bounds(const double* b) {
    if (!b) return CallerBounds{0, 0.0, 0.0, 0.0, 0.0};
    return CallerBounds{1, b[0], b[1], b[2], b[3]};
}

void launch_morton_gpuref(hipStream_t s, const float* xs, const float* ys, const float* ms,
                          const uint32_t* ids, uint32_t n, float4* partials, BuildParams* prm,
                          int depth, uint32_t* status, uint32_t* keys, uint32_t* vals, float4* pk) {
    const uint32_t g = bounds_grid(n);
    k_bounds_partial<<<g, kBlock, 0, s>>>(xs, ys, n, partials);
    k_bounds_final<<<1, kBlock, 0, s>>>(partials, g, n, prm, kTreeGpuRef, caller_bounds(nullptr),
                                        status);
    k_morton_gpuref<<<div_up(n, kBlock), kBlock, 0, s>>>(xs, ys, ms, ids, n, prm, depth, keys,
                                                         vals, pk);
}

// 4 particles per thread above kMortonWide: fewer blocks to repeat the bounds' last step
constexpr uint32_t kMortonWide = 1u << 18;
// up to here every block reads all positions for the bounds (16 loads a thread): no partials launch
constexpr uint32_t kMortonAlone = 4096;

void launch_morton(hipStream_t s, const float* xs, const float* ys, const float* ms,
                   const uint32_t* ids, uint32_t n, float4* partials, BuildParams* prm,
                   uint32_t tree_mode, const double* caller, uint32_t* status, int B, void* keys,
                   uint32_t* vals, bool wide, float4* pk, uint32_t have_partials) {
    const uint32_t nb = n <= kMortonAlone ? 0u : have_partials ? have_partials : bounds_grid(n);
    if (nb && !have_partials) k_bounds_partial<<<nb, kBlock, 0, s>>>(xs, ys, n, partials);
    const CallerBounds cb = caller_bounds(caller);
#define BH_MORTON(K, I)                                                                           \
    k_morton<K, I><<<div_up(n, kBlock * I), kBlock, 0, s>>>(                                      \
        xs, ys, ms, ids, n, partials, nb, tree_mode, cb, prm, status, B, (K*)keys, vals, pk)
    if (n <= kMortonWide) {
        if (wide) BH_MORTON(uint64_t, 1); else BH_MORTON(uint32_t, 1);
    } else {
        if (wide) BH_MORTON(uint64_t, 4); else BH_MORTON(uint32_t, 4);
    }
#undef BH_MORTON
}

uint32_t scan_partials_size(uint64_t n) { return div_up(n, kScanTile) + 1; }

void launch_exclusive_scan(hipStream_t s, const uint32_t* in, uint32_t* out, uint32_t n,
                           uint32_t* partials, uint32_t* total) {
    const uint32_t nb = div_up(n, kScanTile);
    k_scan_reduce<<<nb, kBlock, 0, s>>>(in, n, partials);
    k_scan_partials<<<1, kBlock, 0, s>>>(partials, nb, total);
    k_scan_down<<<nb, kBlock, 0, s>>>(in, out, n, partials);
}

static int sort_items(uint32_t n) { return n <= kSortSmallMax ? kSortItemsSmall : kSortItemsLarge; }

uint32_t sort_blocks(uint32_t n) { return div_up(n, sort_tile(sort_items(n))); }

// radix sort: counts [8][256][tiles] + look-back words [8][tiles][256] + totals [8][256] + tickets;
// bucket sort: ids (2 bytes per key) + look-back words [tiles][buckets] + ticket + sample and
// splitter keys and positions, bucket starts. The largest tile count of any n' <= n.
uint64_t sort_scratch_words(uint32_t n) {
    const uint32_t tiles = max(sort_blocks(n), div_up(min(n, kSortSmallMax), sort_tile(kSortItemsSmall)));
    return 2ull * kSortMaxPasses * 256 * tiles + kSortMaxPasses * 256 + 16 +
           3ull * kBucketSamples + 4ull * kBucketMax;
}

// Mean bucket of a sort, a quarter of what its sorting block holds in LDS: the smaller one leaves
// more buckets to share a small sort (20k keys: 40 blocks), the larger keeps the splitters of a
// large one few (and the runs that a tile writes long).
static uint32_t bucket_mean(uint32_t n) { return n <= (1u << 19) ? 512 : 1024; }
static_assert(kBucketSortMax <= 1024u * kBucketMax && (1u << 19) <= 512u * kBucketMax, "buckets");

// Samples per bucket, a power of two: 4096 keys together, within 8 .. 64 a bucket. Few samples leave
// uneven buckets, and the largest one is the sort's last wave (20k keys: 17 us of k_bucket_sort
// with 8, 12 with 64); ranking 8192 instead of 4096 costs 4 us more.
static uint32_t bucket_sample(uint32_t buckets) {
    uint32_t per = 8;
    while (per < 64 && buckets * per * 2 <= 4096) per *= 2;
    return per;
}

template <typename K>
static void bucket_sort(hipStream_t s, K* keys_a, uint32_t* vals_a, K* keys_b, uint32_t* vals_b,
                        uint32_t n, uint32_t* scratch, uint32_t* err, uint32_t spin_limit) {
    const uint32_t nt = sort_blocks(n), mean = bucket_mean(n), buckets = div_up(n, mean);
    const uint32_t per = bucket_sample(buckets);
    const uint32_t samples = buckets * per;
    uint16_t* id = (uint16_t*)scratch;
    uint32_t* status = scratch + (size_t)kSortMaxPasses * 256 * nt;
    uint32_t* ticket = status + (size_t)kSortMaxPasses * 256 * nt;
    K* sample_key = (K*)(ticket + 16);
    K* split_key = sample_key + kBucketSamples;
    uint32_t* sample_pos = (uint32_t*)(split_key + kBucketMax);
    uint32_t* split_pos = sample_pos + kBucketSamples;
    uint32_t* starts = split_pos + kBucketMax;
    k_bucket_prepare<K><<<div_up(samples, kBlock), kBlock, 0, s>>>(
        keys_a, n, samples, sample_key, sample_pos, status, nt * buckets, ticket);
    k_rank_sort<K, true><<<div_up(samples, kWave), kRankWaves * kWave, 0, s>>>(
        sample_key, sample_pos, samples, per, split_key, split_pos);
#define BH_SPREAD(T)                                                                              \
    k_bucket_count<K, T><<<nt, T, 0, s>>>(keys_a, n, buckets, split_key, split_pos, id, status,   \
                                          ticket, err, spin_limit);                               \
    k_bucket_scatter<K, T><<<nt, T, 0, s>>>(keys_a, vals_a, n, buckets, id, status, err, keys_b,  \
                                            vals_b, starts)
    if (sort_items(n) == kSortItemsSmall) { BH_SPREAD(512); } else { BH_SPREAD(1024); }
#undef BH_SPREAD
    static_assert(kBucketItems * 512 == sort_tile(kSortItemsSmall) &&
                  kBucketItems * 1024 == sort_tile(kSortItemsLarge), "tiles match");
#define BH_SORT(T)                                                                                \
    k_bucket_sort<K, T><<<buckets, T, 0, s>>>(keys_b, vals_b, n, buckets, starts, err, keys_a, \
                                                 vals_a)
    if (mean == 512) BH_SORT(256); else BH_SORT(512);
#undef BH_SORT
}

void launch_sort(hipStream_t s, void* keys_a, uint32_t* vals_a, void* keys_b, uint32_t* vals_b,
                 uint32_t n, int key_bits, bool wide, uint32_t* scratch, uint32_t* err,
                 uint32_t spin_limit, bool* result_in_b) {
    if (n <= kRankSortMax) {
        const dim3 g(div_up(n, kWave)), t(kRankWaves * kWave);
        if (wide)
            k_rank_sort<uint64_t, false><<<g, t, 0, s>>>((const uint64_t*)keys_a, vals_a, n, 1,
                                                         (uint64_t*)keys_b, vals_b);
        else
            k_rank_sort<uint32_t, false><<<g, t, 0, s>>>((const uint32_t*)keys_a, vals_a, n, 1,
                                                         (uint32_t*)keys_b, vals_b);
        *result_in_b = true;
        return;
    }
    if (n <= kBucketSortMax) {
        if (wide)
            bucket_sort<uint64_t>(s, (uint64_t*)keys_a, vals_a, (uint64_t*)keys_b, vals_b, n,
                                  scratch, err, spin_limit);
        else
            bucket_sort<uint32_t>(s, (uint32_t*)keys_a, vals_a, (uint32_t*)keys_b, vals_b, n,
                                  scratch, err, spin_limit);
        *result_in_b = false;
        return;
    }
    const uint32_t nt = sort_blocks(n);
    const int passes = (key_bits + 7) / 8;
    uint32_t* counts = scratch;
    uint32_t* status = counts + (size_t)kSortMaxPasses * 256 * nt;
    uint32_t* totals = status + (size_t)kSortMaxPasses * 256 * nt;
    uint32_t* tickets = totals + kSortMaxPasses * 256;
#define BH_COUNTS(K, T, I)                                                                        \
    k_radix_counts<K, T, I><<<nt, T, 0, s>>>((const K*)keys_a, n, passes, nt, counts, status)
    if (wide) BH_COUNTS(uint64_t, 1024, 4); else BH_COUNTS(uint32_t, 1024, 4);
#undef BH_COUNTS
    k_radix_totals<<<div_up(passes * 256, kWavesPerBlock), kBlock, 0, s>>>(counts, nt, passes,
                                                                            totals, tickets);
    void* kin = keys_a;
    uint32_t* vin = vals_a;
    void* kout = keys_b;
    uint32_t* vout = vals_b;
    for (int p = 0; p < passes; ++p) {
        uint32_t* st = status + (size_t)p * nt * 256;
        const uint32_t* tp = totals + p * 256;
#define BH_PASS(K, T, I)                                                                          \
    k_radix_pass<K, T, I><<<nt, T, 0, s>>>((const K*)kin, vin, (K*)kout, vout, n, 8 * p, tp, st,  \
                                           tickets + p, err, spin_limit)
        static_assert(kSortItemsLarge * kBlock == 1024 * 4 && kBucketSortMax >= kSortSmallMax,
                      "pass tiles match the counting tiles");
        if (wide) BH_PASS(uint64_t, 1024, 4); else BH_PASS(uint32_t, 1024, 4);
#undef BH_PASS
        void* tk = kin; kin = kout; kout = tk;
        uint32_t* tv = vin; vin = vout; vout = tv;
    }
    *result_in_b = (passes & 1) != 0;
}

// Up to here (8,388,608 particles) every block of k_tree_emit_heads adds up the counts of the tiles
// before its own, which spares a build three launches; those reads grow with the square of the tiles,
// so larger builds scan the counts first. The tree's launches, adding / scanning, us: 1M particles
// 30 / 37, 4M 93 / 97, 8M 200 / 196, 17M 473 / 439, 67M 2,373 / 1,895, 134M 5,877 / 4,073, 268M
// 16,135 / 9,199.
constexpr uint32_t kTreeSumsAlone = 8192;

uint32_t tree_sums_words(uint32_t n) {  // counts; then the nodes before each tile, scan partials
    const uint32_t t = div_up(n, kTreeTile);
    return t <= kTreeSumsAlone ? t : 2 * t + scan_partials_size(t);
}

void launch_gather_levels(hipStream_t s, const uint32_t* perm, const float4* pk, const float* vx,
                          const float* vy, float* xo, float* yo, float* mo, float* vxo, float* vyo,
                          uint32_t* ido, float4* pos4, void* codes, bool wide, uint32_t n, int B,
                          int cap, int fixed_depth, uint8_t* lcp1, uint32_t* cnt,
                          uint32_t* sums, int R, const uint32_t* status) {
#define BH_LEVELS(K)                                                                              \
    k_gather_levels<K><<<div_up(n, kTreeTile), kTreeTile, 0, s>>>(                                \
        perm, pk, vx, vy, xo, yo, mo, vxo, vyo, ido, pos4, (K*)codes, n, B, R, cap, fixed_depth,  \
        lcp1, cnt, sums, status)
    if (wide) BH_LEVELS(uint64_t); else BH_LEVELS(uint32_t);
#undef BH_LEVELS
}

void launch_tree(hipStream_t s, const void* codes, bool wide, uint32_t n, int B,
                 int single_child_pp, const uint8_t* lcp1, const uint32_t* cnt, uint32_t* noff,
                 uint32_t* sums, BuildParams* prm, Node* nodes, uint32_t* child4,
                 uint32_t cap_nodes, int R, const BuildParams* sys_prm) {
    const uint32_t g = div_up(n, kTreeTile), gn = div_up(cap_nodes, kTreeThreads);
#define BH_NODES(K)                                                                               \
    k_tree_emit_nodes<K><<<gn, kTreeThreads, 0, s>>>((const K*)codes, n, B, R, lcp1, noff, prm,   \
                                                     sys_prm, single_child_pp, nodes, child4,     \
                                                     cap_nodes)
    const bool scan = g > kTreeSumsAlone;
    if (scan) launch_exclusive_scan(s, sums, sums + g, g, sums + 2 * (size_t)g, nullptr);
    k_tree_emit_heads<<<g, kTreeTile, 0, s>>>(n, lcp1, cnt, scan ? sums + g : sums, scan ? 1 : 0,
                                              noff, prm, nodes, (uint4*)child4, cap_nodes);
    if (wide) BH_NODES(uint64_t); else BH_NODES(uint32_t);
#undef BH_NODES
}

void launch_bounds_batched(hipStream_t s, const float* xs, const float* ys, const uint2* blk,
                           uint32_t nblk, const uint32_t* blk_off, const uint32_t* sys_off,
                           uint32_t nsys, float4* partials, BuildParams* sys_prm,
                           BuildParams* prm, uint32_t* status) {
    k_bounds_seg_partial<<<nblk, kBlock, 0, s>>>(xs, ys, blk, partials);
    k_bounds_seg_final<<<nsys, kBlock, 0, s>>>(partials, blk_off, sys_off, sys_prm, prm, status);
}

void launch_morton_batched(hipStream_t s, const float* xs, const float* ys, const float* ms,
                           const uint32_t* ids, uint32_t n, const uint32_t* sys_off, uint32_t nsys,
                           const BuildParams* sys_prm, int B, uint64_t* keys, uint32_t* vals,
                           float4* pk) {
    k_morton_seg<<<div_up(n, kBlock), kBlock, 0, s>>>(xs, ys, ms, ids, n, sys_off, nsys, sys_prm, B,
                                                      keys, vals, pk);
}

void launch_batch_roots(hipStream_t s, const uint32_t* sys_off, uint32_t nsys,
                        const uint32_t* noff, const BuildParams* prm, uint32_t* roots) {
    k_batch_roots<<<div_up(nsys, kBlock), kBlock, 0, s>>>(sys_off, nsys, noff, prm, roots);
}

uint32_t up_chunks(uint32_t cap_nodes) { return div_up(cap_nodes, kUpChunkSmall); }

// Chunks of 512 nodes up to kUpSmallMax points: with 2048, 70k points are 20 blocks. Larger trees take
// 2048, so that the nodes left to k_up_top (up to one per level and chunk) fit its LDS at 1M.
void launch_upward(hipStream_t s, const float4* pos4, Node* nodes, const uint32_t* child4,
                   float4* m2, const BuildParams* prm, uint32_t* deferred, uint32_t* bylevel,
                   uint32_t cap_nodes, uint32_t n, bool big_leaves) {
    const bool small = n <= kUpSmallMax;
    const uint32_t chunk = small ? kUpChunkSmall : kUpChunk;
    const uint32_t nch = div_up(cap_nodes, chunk);
    const bool big_done = big_leaves && !m2;
    if (big_done)
        k_big_leaf_moments<<<div_up(cap_nodes, kWavesPerBlock), kBlock, 0, s>>>(pos4, nodes, prm,
                                                                                cap_nodes);
#define BH_UP(M2)                                                                                 \
    if (small)                                                                                    \
        k_up_chunk<kUpChunkSmall, kUpChunkSmall, M2><<<nch, kUpChunkSmall, 0, s>>>(               \
            pos4, nodes, (const uint4*)child4, m2, prm, deferred, cap_nodes, big_done ? 1 : 0);   \
    else                                                                                          \
        k_up_chunk<kUpChunk, kUpThreads, M2><<<nch, kUpThreads, 0, s>>>(                          \
            pos4, nodes, (const uint4*)child4, m2, prm, deferred, cap_nodes, big_done ? 1 : 0);   \
    k_up_top<M2><<<1, kUpThreads, 0, s>>>(nodes, (const uint4*)child4, m2, prm, deferred,         \
                                          bylevel, nch, chunk, cap_nodes)
    if (m2) {
        BH_UP(true);
    } else {
        BH_UP(false);
    }
#undef BH_UP
}

void launch_tree_stats(hipStream_t s, const Node* nodes, const BuildParams* prm,
                       uint32_t cap_nodes, int depth_limit, uint32_t leaf_cap, uint2* out,
                       uint32_t blocks) {
    k_tree_stats<<<blocks, kBlock, 0, s>>>(nodes, prm, cap_nodes, depth_limit, leaf_cap, out);
}

void launch_fill_u32(hipStream_t s, uint32_t* p, uint64_t n, uint32_t v) {
    if (n) k_fill_u32<<<div_up(n, kBlock), kBlock, 0, s>>>(p, n, v);
}

void launch_fill_f32(hipStream_t s, float* p, uint64_t n, float v) {
    union {
        float f;
        uint32_t u;
    } c;
    c.f = v;
    launch_fill_u32(s, (uint32_t*)p, n, c.u);
}

void launch_init_state(hipStream_t s, uint32_t n, uint32_t* id, float* m, float* vx, float* vy) {
    if (n) k_init_state<<<div_up(n, kBlock), kBlock, 0, s>>>(n, id, m, vx, vy);
}

void launch_tree_slots(hipStream_t s, const uint32_t* codes, const Node* nodes,
                       const BuildParams* prm, uint32_t cap_nodes, int depth, uint32_t* first_child,
                       uint32_t* first_particle, uint32_t* count, uint64_t slots) {
    k_clear_slots<<<div_up(slots, kBlock), kBlock, 0, s>>>(first_child, first_particle, count,
                                                           slots);
    k_tree_slots<<<div_up(cap_nodes, kBlock), kBlock, 0, s>>>(codes, nodes, prm, cap_nodes, depth,
                                                              first_child, first_particle, count);
}

}  // namespace bh
