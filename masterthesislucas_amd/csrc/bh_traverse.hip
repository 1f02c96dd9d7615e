// Barnes-Hut traversal on gfx950: one wave = 64 Morton-consecutive sink particles that walk the
// pre-order tree together (k_walk below), each particle with exactly the per-particle Barnes-Hut
// decisions of the reference traversal (nBodySolverBH.h:56-89 /
// nBodySolverFMM_SYM_MORTON.h:272-313). Near-field cells are summed particle by particle with the
// self term excluded by index. Forces accumulate in FP32 with Kahan compensation.
#include "bh_common.h"
#include "bh_launch.h"
#include "bh_mlp.h"

#include <type_traits>


namespace bh {

__device__ __forceinline__ void kahan_add(float& s, float& c, float v) {
    const float y = v - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
}

// a wave-uniform value moved to a scalar register
__device__ __forceinline__ uint32_t uniform_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ float uniform_f32(float v) {
    return __uint_as_float(uniform_u32(__float_as_uint(v)));
}

// Node record as raw bits (cx, cy, mass, l2 | skip, first, count, meta)
struct NodeBits {
    uint4 a, b;
    __device__ __forceinline__ float cx() const { return __uint_as_float(a.x); }
    __device__ __forceinline__ float cy() const { return __uint_as_float(a.y); }
    __device__ __forceinline__ float mass() const { return __uint_as_float(a.z); }
    __device__ __forceinline__ float l2() const { return __uint_as_float(a.w); }
    __device__ __forceinline__ uint32_t skip() const { return b.x; }
    __device__ __forceinline__ uint32_t first() const { return b.y; }
    __device__ __forceinline__ uint32_t count() const { return b.z; }
    __device__ __forceinline__ uint32_t meta() const { return b.w; }
};
__device__ __forceinline__ NodeBits load_node(const Node* __restrict__ nodes, uint32_t k) {
    const uint4* p = reinterpret_cast<const uint4*>(nodes + k);
    return NodeBits{p[0], p[1]};
}
// ------------------------------------------------------------------------------------------
// The walk.
//
// One wave holds 64 Morton-consecutive sinks, one per lane, and their bounding box. It keeps a
// stack of opened cells in LDS, each with the mask of the lanes that opened it. A step takes up
// to kWalkPop cells off the stack and loads the records of their children, one per lane, so a
// step's 64 nodes cost one memory round trip instead of one each. Every child is then judged
// against the box: with dmin and dmax the squared distances from its centre of mass to the
// nearest and farthest edges, evaluated like a lane's own d2 (subtraction, square and fma are
// monotone under rounding), every lane's d2 lies in [dmin, dmax], so dmin > lim proves that all
// lanes accept the cell and dmax <= lim that none does. Only the cells in between are tested lane
// by lane (about a sixth of the visits on a disk at theta = 0.5). Each particle sees exactly the
// decisions of the per-particle rule.
//
// Accepted cells are summed from LDS broadcasts, those that every lane accepts without a mask,
// the others under the lanes' exec mask. Particle-particle cells are collected, their sources
// staged through LDS 64 at a time whatever the cells' sizes, and summed under each cell's mask;
// the sink itself can only be among the sources of a cell that holds some of the wave's own
// sinks, and only those cells compare indices.
//
// Sums. Every sink has kWalkParts compensated sums; entry i of a step's accepted cells and source
// i of a particle-particle cell belong to part i % kWalkParts, and the parts are added in order,
// with compensation, at the end. A part's plain sums are folded into its compensated ones after at
// most 8 cells or 16 sources (error against FP64 sums of the same interactions: 2.8e-8 rms of the summed
// magnitudes on the two disks, as before). Because the parts are fixed, 1, 2 or 4 waves can share a sink group (NP = 4, 2 or 1
// parts per wave: they all take the same path and add only their parts) with bit-identical
// results: launches with too few sink groups to fill the device use more waves per group
// (walk_waves_per_group). A particle-particle cell of more than kWalkGiant points, gravity (a cell
// with one child is one, and can hold a whole cluster), is one plain sum over its sources in
// order, added to part 0: the rounding of so long a plain sum can exceed the rest of a sink's
// error by far (half of 1M points in one cell: 0.6%), so its order is part of the result and
// stays what it has always been. Telling such cells apart costs 0.5% of a walk without them; a
// walk over one with 524,288 points 331 -> 258 ms.
//
// Results go to sorted order and, where the call returns them, to the caller's order too: the
// scattered stores cost nothing beside the sums, a launch of their own 4 us at 2,000 sinks, 24 at
// 1M and 168 at 4M.
//
// Bound by VALU issue (13 slots per interaction, the reciprocal square root counting as four)
// where the waves fill the device, by the latency of the steps where they do not. Measured
// against the former walk (one node per visit for 128 sinks, fetched with scalar loads one visit
// ahead; every lane tested every node):
//   two disks, theta 0.5, 1,048,576 sinks    851 -> 654 us
//                            200,003 sinks   424 -> 200 us
//   uniform disk, 2,000 sinks                125 ->  55 us
//   t-SNE, 70,000 points                     268 (spread) / 325 (compact) -> 110 / 140 us
//   128 systems of 1,024 to 65,536           1080 -> 778 us
// ------------------------------------------------------------------------------------------
constexpr int kWalkParts = 4;
constexpr int kWalkStack = 192;              // opened cells
constexpr int kWalkPop = 16;                 // cells opened per step (4 children each)
constexpr int kWalkDeep = 3 * kMaxLevels;    // entries a depth-first descent can add to the stack
constexpr int kWalkCells = 96;               // particle-particle cells waiting
constexpr int kWalkFlush = kWalkCells - 64;  // summed above this many (a step adds at most 64)
constexpr uint32_t kWalkFold = 16;           // terms of a part's plain sum
constexpr uint32_t kWalkGiant = 4096;        // points of a cell that is summed by itself
static_assert(kWalkStack >= kWalkDeep + 4 * kWalkPop, "room for a bulk step and a descent");

struct __attribute__((aligned(16))) WalkLds {  // per wave
    float4 rec[kWave];          // the step's cells (x, y, mass, limit), then sources
    uint4 cells[kWalkCells];    // first source, count, lane mask
    uint2 mask[kWalkStack];
    uint32_t node[kWalkStack];
};
struct WalkLdsLearned : WalkLds {
    uint2 slot[kWave];  // the step's cells: node, l2 / band2
};

__device__ __forceinline__ void wave_lds_sync() {  // LDS of this wave only: order, no wait
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint32_t lane_read(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
__device__ __forceinline__ uint64_t lane_read2(uint32_t lo, uint32_t hi, uint32_t lane) {
    return ((uint64_t)lane_read(hi, lane) << 32) | lane_read(lo, lane);
}

template <bool TOT>
struct WalkSum {  // one part: plain sums (b) and compensated ones (a with terms c)
    float bx = 0.f, by = 0.f, bt = 0.f;
    float ax = 0.f, cx = 0.f, ay = 0.f, cy = 0.f, at = 0.f, ct = 0.f;
    __device__ __forceinline__ void fold() {
        kahan_add(ax, cx, bx);
        kahan_add(ay, cy, by);
        if (TOT) kahan_add(at, ct, bt);
        bx = by = bt = 0.f;
    }
};

// gravity: a += m (q - p) / (|q - p|^2 + eps^2)^(3/2); potential -= m / sqrt(...)
// t-SNE:   w = 1 / (1 + |p - q|^2); total += m w; derivative += m w^2 (p - q)
// Every multiply-add is written as one: left to the compiler, the potential's was fused in the plain walk
// and not in the learned one, and their potentials differed by 1e-10.
template <int KERNEL, bool TOT>
__device__ __forceinline__ void walk_pair(WalkSum<TOT>& s, float dx, float dy, float m,
                                          float eps2) {
    if (KERNEL == kKernelGravity) {
        const float inv = __builtin_amdgcn_rsqf(fmaf(dx, dx, fmaf(dy, dy, eps2)));
        const float mi = m * inv;
        const float f = mi * inv * inv;
        s.bx = fmaf(f, dx, s.bx);
        s.by = fmaf(f, dy, s.by);
        if (TOT) s.bt = fmaf(-m, inv, s.bt);
    } else {
        const float w = __builtin_amdgcn_rcpf(fmaf(dx, dx, fmaf(dy, dy, 1.0f)));
        const float mw = m * w;
        const float f = mw * w;
        s.bx = fmaf(-f, dx, s.bx);
        s.by = fmaf(-f, dy, s.by);
        if (TOT) s.bt = fmaf(m, w, s.bt);
    }
}

// Learned far-field correction inside the walk (LTERMS = 3 or 7 basis terms; 0: none): each
// accepted cell whose l / r is at least `band` (all accepted cells when inv_band2 = 0) gets its
// monopole corrected by (M l^2 / r^4) sum_j c_j b_j(d / r, l / r), with the cell's coefficient
// record (kCoefStride floats, computed once per cell and build by the network) read by the wave
// with scalar loads.
struct LearnArgs {
    const float4* coef = nullptr;
    float inv_band2 = 0.f;
};

// RES: waves per SIMD that the registers must allow (walk_resident)
template <int KERNEL, bool TOT, int NP, bool BATCHED, int LTERMS, int RES>
__global__ __launch_bounds__(kBlock, RES) void k_walk(const float4* __restrict__ pos4,
                                                 const Node* __restrict__ nodes,
                                                 const uint32_t* __restrict__ child4,
                                                 const BuildParams* __restrict__ prm, uint32_t n,
                                                 float inv_theta2, float eps2, float scale,
                                                 float* __restrict__ ax_out,
                                                 float* __restrict__ ay_out,
                                                 float* __restrict__ tot_out,
                                                 unsigned long long* __restrict__ counters,
                                                 TraverseBatch batch, LearnArgs la,
                                                 CallerOut out) {
    constexpr int kGroupWaves = kWalkParts / NP;  // waves per sink group
    static_assert(kWavesPerBlock % kGroupWaves == 0, "whole groups per block");
    using Lds = std::conditional_t<LTERMS != 0, WalkLdsLearned, WalkLds>;
    __shared__ Lds lds[kWavesPerBlock];
    const uint32_t lane = threadIdx.x & 63;
    // wave-uniform (the compiler cannot tell that threadIdx.x / 64 is)
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t p0 = (w % kGroupWaves) * NP;  // first part of this wave
    const uint32_t group = blockIdx.x * (kWavesPerBlock / kGroupWaves) + w / kGroupWaves;
    Lds& L = lds[w];
    const uint64_t lt = lane_mask_lt();

    uint32_t base = group * kWave, count, k0 = 0, slice = 0;
    bool any;
    if constexpr (BATCHED) {
        base = count = 0;
        any = false;
        if (group < batch.n_work) {
            const uint4 wk = batch.work[group];
            k0 = batch.roots[wk.z];
            if (k0 != kNone) {
                base = wk.x;
                count = wk.y;
                slice = wk.w;
                any = true;
            }
        }
        base = uniform_u32(base);
        count = uniform_u32(count);
        slice = uniform_u32(slice);
        k0 = uniform_u32(k0);
    } else {
        count = n > base ? min(n - base, (uint32_t)kWave) : 0u;
        any = count != 0u && prm->n_nodes != 0u;
    }
    any = uniform_u32(any ? 1u : 0u) != 0u;
    const uint32_t idx = base + lane;
    const bool valid = lane < count;
    const float4 me = valid ? pos4[idx] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float px = me.x, py = me.y;
    const uint64_t full = __ballot(valid);
    float xlo = valid ? px : INFINITY, xhi = valid ? px : -INFINITY;
    float ylo = valid ? py : INFINITY, yhi = valid ? py : -INFINITY;
    for (int o = 32; o > 0; o >>= 1) {
        xlo = fminf(xlo, __shfl_xor(xlo, o, kWave));
        xhi = fmaxf(xhi, __shfl_xor(xhi, o, kWave));
        ylo = fminf(ylo, __shfl_xor(ylo, o, kWave));
        yhi = fmaxf(yhi, __shfl_xor(yhi, o, kWave));
    }
    xlo = uniform_f32(xlo);
    xhi = uniform_f32(xhi);
    ylo = uniform_f32(ylo);
    yhi = uniform_f32(yhi);
    // BATCHED slice of a heavy entry: this wave adds every sF-th step's cells and every sF-th
    // block of sources, from the sf-th on
    const uint32_t sf = slice & 15u, sF = slice ? (slice >> 4) & 15u : 1u;

    WalkSum<TOT> sum[NP];
    uint32_t terms = 0;  // terms of the parts' plain sums (cells count as two)
    auto fold_all = [&]() {
#pragma unroll
        for (int p = 0; p < NP; ++p) sum[p].fold();
        terms = 0;
    };
    uint32_t n_pn = 0;  // per lane: interactions of the nodes it judged
    uint64_t n_pp = 0;
    int sp = 0, nc = 0;
    uint32_t blk_no = sf == 0 ? 0u : sF - sf, step_no = blk_no;  // 0 (mod sF): this wave's turn

    // particle-particle sums over the collected cells
    auto flush = [&]() {
        for (int c0 = 0; c0 < nc; c0 += kWave) {
            const int nn = min(nc - c0, kWave);
            const uint4 cell = (int)lane < nn ? L.cells[c0 + lane] : make_uint4(0, 0, 0, 0);
            // the ordinary cells, then the giant ones each by itself
            uint64_t giants = __ballot(KERNEL == kKernelGravity && cell.y > kWalkGiant);
            uint32_t giant = kNone;
            bool now = KERNEL != kKernelGravity || cell.y <= kWalkGiant;
            for (;;) {
                const uint32_t cr = now ? (cell.y + 3u) & ~3u : 0u;  // slots: whole quads
                uint32_t end = cr;
                for (int o = 1; o < kWave; o <<= 1) {
                    const uint32_t t = __shfl_up(end, o, kWave);
                    if ((int)lane >= o) end += t;
                }
                const uint32_t off = end - cr, stop = off + cell.y;
                const bool own = cell.x < base + count && base < cell.x + cell.y;
                const uint32_t total = lane_read(end, kWave - 1);
                // the source of this lane's slot in the 64 slots from `blk` on; the slots past a
                // cell's last source repeat it
                auto fetch = [&](uint32_t blk) {
                    uint32_t src = 0;
                    uint64_t m = __ballot(end > blk && off < blk + kWave && cr != 0u);
                    while (m) {
                        const uint32_t e = (uint32_t)__builtin_ctzll(m);
                        m &= m - 1;
                        const uint32_t o = lane_read(off, e);
                        // (computed for every lane: an expression inside the selection is hoisted
                        // by the compiler with the selection's condition taken for granted)
                        const uint32_t at = lane_read(cell.x, e) +
                                            min(blk + lane - o, lane_read(cell.y, e) - 1u);
                        src = blk + lane >= o ? at : src;
                    }
                    return pos4[src];
                };
                float4 q = fetch(0);
                for (uint32_t blk = 0; blk < total; blk += kWave) {
                    const bool mine = !BATCHED || blk_no == 0u;
                    if constexpr (BATCHED) blk_no = blk_no + 1u == sF ? 0u : blk_no + 1u;
                    wave_lds_sync();
                    L.rec[lane] = q;
                    wave_lds_sync();
                    if (blk + kWave < total) q = fetch(blk + kWave);  // in flight during the sums
                    if (!mine) continue;
                    if (giant != kNone) {  // one cell in order, in one plain sum
                        if (p0 != 0) continue;
                        const uint32_t b = min(lane_read(cell.y, giant) - blk, (uint32_t)kWave);
                        const int s0 = (int)(base - lane_read(cell.x, giant) - blk);  // first sink
                        const uint64_t msk = lane_read2(cell.z, cell.w, giant);
                        if (!__builtin_amdgcn_inverse_ballot_w64(msk)) continue;
                        if (s0 >= (int)b || s0 + (int)count <= 0) {
                            uint32_t j = 0;
                            for (; j + 4 <= b; j += 4) {
                                float4 s[4];
#pragma unroll
                                for (int t = 0; t < 4; ++t) s[t] = L.rec[j + t];
#pragma unroll
                                for (int t = 0; t < 4; ++t)
                                    walk_pair<KERNEL, TOT>(sum[0], s[t].x - px, s[t].y - py, s[t].z,
                                                           eps2);
                            }
                            for (; j < b; ++j)
                                walk_pair<KERNEL, TOT>(sum[0], L.rec[j].x - px, L.rec[j].y - py,
                                                       L.rec[j].z, eps2);
                        } else {
                            for (uint32_t j = 0; j < b; ++j)
                                if ((int)j != s0 + (int)lane)
                                    walk_pair<KERNEL, TOT>(sum[0], L.rec[j].x - px, L.rec[j].y - py,
                                                           L.rec[j].z, eps2);
                        }
                        continue;
                    }
                    // cells without sinks of this wave, then those that hold some
                    const bool here = stop > blk && off < blk + kWave && cr != 0u;
                    const uint32_t from = max(off, blk) - blk, to = min(stop - blk, (uint32_t)kWave);
                    uint64_t m = __ballot(here && !own);
                    while (m) {
                        const uint32_t e = (uint32_t)__builtin_ctzll(m);
                        m &= m - 1;
                        uint32_t j = lane_read(from, e);  // a multiple of 4
                        const uint32_t b = lane_read(to, e);
                        const uint64_t msk = lane_read2(cell.z, cell.w, e);
                        const uint32_t quads = (b - j + 3u) >> 2;
                        if (terms + quads > kWalkFold) fold_all();
                        terms += quads;
                        if (__builtin_amdgcn_inverse_ballot_w64(msk)) {
                            for (; j + 4 <= b; j += 4) {
                                float4 s[NP];
#pragma unroll
                                for (int p = 0; p < NP; ++p) s[p] = L.rec[j + p0 + p];
#pragma unroll
                                for (int p = 0; p < NP; ++p)
                                    walk_pair<KERNEL, TOT>(sum[p], s[p].x - px, s[p].y - py, s[p].z,
                                                           eps2);
                            }
#pragma unroll
                            for (int p = 0; p < NP; ++p)
                                if (j + p0 + p < b) {
                                    const float4 s = L.rec[j + p0 + p];
                                    walk_pair<KERNEL, TOT>(sum[p], s.x - px, s.y - py, s.z, eps2);
                                }
                        }
                    }
                    m = __ballot(here && own);
                    while (m) {
                        const uint32_t e = (uint32_t)__builtin_ctzll(m);
                        m &= m - 1;
                        uint32_t j = lane_read(from, e);
                        const uint32_t b = lane_read(to, e);
                        const uint64_t msk = lane_read2(cell.z, cell.w, e);
                        // slot of the sink itself in this block
                        const uint32_t self = idx - lane_read(cell.x, e) + lane_read(off, e) - blk;
                        const uint32_t quads = (b - j + 3u) >> 2;
                        if (terms + quads > kWalkFold) fold_all();
                        terms += quads;
                        if (__builtin_amdgcn_inverse_ballot_w64(msk)) {
                            for (; j < b; j += 4)
#pragma unroll
                                for (int p = 0; p < NP; ++p) {
                                    const uint32_t jj = j + p0 + p;
                                    if (jj < b && jj != self) {
                                        const float4 s = L.rec[jj];
                                        walk_pair<KERNEL, TOT>(sum[p], s.x - px, s.y - py, s.z, eps2);
                                    }
                                }
                        }
                    }
                }
                if (giant != kNone) fold_all();
                if (!giants) break;
                giant = (uint32_t)__builtin_ctzll(giants);
                giants &= giants - 1;
                now = lane == giant;
                fold_all();
            }
        }
        wave_lds_sync();
        nc = 0;
    };

    uint32_t id = kNone;
    // one accepted cell (staged at slot e) for the calling lanes. Its index and limit come from LDS
    // like its record: the slot's own lane need not be among the callers, and a value read from a
    // lane outside a branch survives a spill or a copy made inside it only by chance. (Both read
    // by v_readlane before the branch: 2.55 -> 2.67 ms for the walk of 4,194,304 sinks.)
    auto cell_pair = [&](WalkSum<TOT>& s, const float4 q, uint32_t e) {
        const float dx = q.x - px, dy = q.y - py;
        if constexpr (LTERMS == 0) {
            walk_pair<KERNEL, TOT>(s, dx, dy, q.z, eps2);
        } else {
            const uint2 sn = L.slot[e];
            walk_pair<KERNEL, TOT>(s, dx, dy, q.z, eps2);
            const float d2 = fmaf(dx, dx, dy * dy);
            const bool corr = la.inv_band2 == 0.f || !(d2 > __uint_as_float(sn.y));
            const float4* cr = la.coef + (size_t)uniform_u32(sn.x) * (kCoefStride / 4);
            const float4 c0 = cr[0], c1 = cr[1], c2 = cr[2], c3 = cr[3];
            if (corr) {
                const float rec[kCoefStride] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w,
                                                c2.x, c2.y, c2.z, c2.w, c3.x, c3.y, c3.z, c3.w};
                float gx, gy;
                learned_correction<LTERMS>(dx, dy, d2, rec, gx, gy);
                s.bx += gx;
                s.by += gy;
            }
        }
    };

    uint32_t mlo = 0, mhi = 0;  // lanes that reach this lane's node
    if (any && lane == 0) {
        id = k0;
        mlo = (uint32_t)full;
        mhi = (uint32_t)(full >> 32);
    }
    while (any) {
        // one node per lane: its record and the box's verdict
        const bool live = id != kNone;
        const NodeBits nd = load_node(nodes, live ? id : k0);
        const float lim = nd.l2() * inv_theta2;
        const float xa = nd.cx() - xlo, xb = nd.cx() - xhi;  // xb <= every lane's dx <= xa
        const float ya = nd.cy() - ylo, yb = nd.cy() - yhi;
        const float nx = fmaxf(fmaxf(xb, -xa), 0.f), ny = fmaxf(fmaxf(yb, -ya), 0.f);
        const float fx = fmaxf(xa, -xb), fy = fmaxf(ya, -yb);
        const bool acc_all = live && fmaf(nx, nx, ny * ny) > lim;
        const bool open_all = live && !acc_all && fmaf(fx, fx, fy * fy) <= lim;
        wave_lds_sync();
        L.rec[lane] = make_float4(nd.cx(), nd.cy(), nd.mass(), lim);
        if constexpr (LTERMS != 0)
            L.slot[lane] = make_uint2(id, __float_as_uint(nd.l2() * la.inv_band2));
        wave_lds_sync();
        uint32_t olo = open_all ? mlo : 0u, ohi = open_all ? mhi : 0u;  // lanes that open it
        uint64_t xm = __ballot(live && !acc_all && !open_all);
        while (xm) {  // lane by lane
            const uint32_t e = (uint32_t)__builtin_ctzll(xm);
            xm &= xm - 1;
            const float4 q = L.rec[e];
            const float dx = q.x - px, dy = q.y - py;
            const float d2 = fmaf(dx, dx, dy * dy);
            const uint64_t op = lane_read2(mlo, mhi, e) & ~__ballot(d2 > q.w);
            olo = lane == e ? (uint32_t)op : olo;
            ohi = lane == e ? (uint32_t)(op >> 32) : ohi;
        }
        const uint32_t alo = mlo & ~olo, ahi = mhi & ~ohi;  // lanes that accept it
        const bool opened = (olo | ohi) != 0u;
        const bool is_pp = (nd.meta() & kMetaPP) != 0u;
        const bool all = live && alo == (uint32_t)full && ahi == (uint32_t)(full >> 32);
        uint64_t am = __ballot(all), mm = __ballot(live && !all && (alo | ahi) != 0u);
        n_pn += (uint32_t)__popc(alo) + (uint32_t)__popc(ahi);
        // particle-particle cells wait, opened cells go on the stack
        const uint64_t cm = __ballot(opened && is_pp), pm = __ballot(opened && !is_pp);
        if (opened && is_pp) {
            L.cells[nc + __popcll(cm & lt)] = make_uint4(nd.first(), nd.count(), olo, ohi);
            n_pp += (uint64_t)((uint32_t)__popc(olo) + (uint32_t)__popc(ohi)) * nd.count();
            if (nd.first() < base + count && base < nd.first() + nd.count()) {
                // sinks of the wave among the sources, a run of lanes, skip themselves
                const uint32_t b0 = max(nd.first(), base) - base;
                const uint32_t b1 = min(nd.first() + nd.count() - base, (uint32_t)kWave);
                const uint64_t run = (~0ull >> (kWave - (b1 - b0))) << b0;
                n_pp -= (uint32_t)__popcll((((uint64_t)ohi << 32) | olo) & run);
            }
        }
        nc += __popcll(cm);
        if (opened && !is_pp) {
            const int at = sp + __popcll(pm & lt);
            L.node[at] = id;
            L.mask[at] = make_uint2(olo, ohi);
        }
        sp += __popcll(pm);
        wave_lds_sync();
        // the next step's cells off the stack, its nodes' indices in flight during the sums. A
        // bulk step leaves room for a depth-first descent (each level adds at most 3), which a
        // nearly full stack falls back to.
        const int room = (kWalkStack - kWalkDeep - sp) / 3;
        const int take = min(sp, max(1, min(kWalkPop, room)));
        sp -= take;
        const uint32_t par = lane >> 2;
        const bool up = (int)par < take;
        const uint32_t pid = up ? L.node[sp + par] : 0u;
        const uint2 pmask = up ? L.mask[sp + par] : make_uint2(0u, 0u);
        const uint32_t next_id = up ? child4[4 * (size_t)pid + (lane & 3)] : kNone;

        const bool mine = !BATCHED || step_no == 0u;
        if constexpr (BATCHED) step_no = step_no + 1u == sF ? 0u : step_no + 1u;
        if (mine) {
            // cells that every lane accepts, four at a time, one per part; what is left over
            // joins the others
            while (__popcll(am) >= kWalkParts) {
                uint32_t e[kWalkParts];
#pragma unroll
                for (int p = 0; p < kWalkParts; ++p) {
                    e[p] = (uint32_t)__builtin_ctzll(am);
                    am &= am - 1;
                }
                if constexpr (NP == 2) {
                    e[0] = p0 ? e[2] : e[0];
                    e[1] = p0 ? e[3] : e[1];
                } else if constexpr (NP == 1) {
                    const uint32_t a = p0 & 1u ? e[1] : e[0], b = p0 & 1u ? e[3] : e[2];
                    e[0] = p0 & 2u ? b : a;
                }
                if (terms + 2 > kWalkFold) fold_all();
                terms += 2;
                float4 q[NP];
#pragma unroll
                for (int p = 0; p < NP; ++p) q[p] = L.rec[e[p]];
#pragma unroll
                for (int p = 0; p < NP; ++p) cell_pair(sum[p], q[p], e[p]);
            }
            mm |= am;
            // cells that some lanes accept
            while (mm) {
                if (terms + 2 > kWalkFold) fold_all();
                terms += 2;
#pragma unroll
                for (int p = 0; p < kWalkParts; ++p) {
                    if (!mm) break;
                    const uint32_t e = (uint32_t)__builtin_ctzll(mm);
                    mm &= mm - 1;
                    if (NP != kWalkParts && ((uint32_t)p < p0 || (uint32_t)p >= p0 + NP)) continue;
                    const float4 q = L.rec[e];
                    const uint64_t msk = lane_read2(alo, ahi, e);
                    if (__builtin_amdgcn_inverse_ballot_w64(msk)) {
                        if constexpr (NP == 1) cell_pair(sum[0], q, e);
                        else if constexpr (NP == 2) cell_pair(sum[p & 1], q, e);
                        else cell_pair(sum[p], q, e);
                    }
                }
            }
        }
        if (nc > kWalkFlush || (take == 0 && nc > 0)) flush();
        if (take == 0) break;
        id = next_id;
        mlo = id != kNone ? pmask.x : 0u;
        mhi = id != kNone ? pmask.y : 0u;
    }
    fold_all();
    // the parts (and their compensation terms), added in order with compensation
    float ox = 0.f, oy = 0.f, ot = 0.f, ex = 0.f, ey = 0.f, et = 0.f;
    auto add_part = [&](float ax, float cx, float ay, float cy, float at, float ct) {
        kahan_add(ox, ex, ax);
        kahan_add(ox, ex, -cx);
        kahan_add(oy, ey, ay);
        kahan_add(oy, ey, -cy);
        if (TOT) kahan_add(ot, et, at);
        if (TOT) kahan_add(ot, et, -ct);
    };
    if constexpr (NP == kWalkParts) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
            add_part(sum[p].ax, sum[p].cx, sum[p].ay, sum[p].cy, sum[p].at, sum[p].ct);
    } else {
        // by the group's first wave, through the LDS of the group's waves
        float* red = reinterpret_cast<float*>(&lds[w - w % kGroupWaves]);
        static_assert(kGroupWaves * sizeof(WalkLds) >= 6 * kWalkParts * kWave * sizeof(float),
                      "room for the parts");
        __syncthreads();
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            float* r = red + 6 * (p0 + p) * kWave + lane;
            r[0 * kWave] = sum[p].ax;
            r[1 * kWave] = sum[p].cx;
            r[2 * kWave] = sum[p].ay;
            r[3 * kWave] = sum[p].cy;
            r[4 * kWave] = sum[p].at;
            r[5 * kWave] = sum[p].ct;
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < kWalkParts; ++p) {
            const float* r = red + 6 * p * kWave + lane;
            add_part(r[0 * kWave], r[1 * kWave], r[2 * kWave], r[3 * kWave], r[4 * kWave],
                     r[5 * kWave]);
        }
    }
    ox -= ex;
    oy -= ey;
    ot -= et;
    const bool writer = NP == kWalkParts || p0 == 0;
    if (writer && valid) {
        if (BATCHED && slice) {  // a heavy entry's slice: partial results
            const size_t plane = (size_t)batch.side_slots * kHeavySlices * kHeavySinks;
            const size_t o = ((size_t)(slice >> 8) * kHeavySlices + sf) * kHeavySinks + lane;
            batch.side[o] = scale * ox;
            batch.side[plane + o] = scale * oy;
            if (TOT) batch.side[2 * plane + o] = scale * ot;
        } else {
            const float sx = scale * ox, sy = scale * oy;
            ax_out[idx] = sx;
            ay_out[idx] = sy;
            if (TOT) tot_out[idx] = scale * ot;
            if (out.id) {  // also in the caller's order, beside other waves' sums
                const uint32_t o = out.id[idx];
                if (out.x) out.x[o] = sx;
                if (out.y) out.y[o] = sy;
            }
        }
    }
    // one pair per wave (no same-address device atomics): the group's first wave counts for it,
    // the first slice for its entry
    const bool counts = writer && sf == 0u;
    const unsigned long long s_pn = wave_sum_u64(counts ? n_pn : 0u);
    const unsigned long long s_pp = wave_sum_u64(counts ? n_pp : 0u);
    if (lane == 0) {
        const size_t gw = (size_t)blockIdx.x * kWavesPerBlock + w;
        counters[2 * gw] = s_pn;
        counters[2 * gw + 1] = s_pp;
    }
}

// ------------------------------------------------------------------------------------------
// The pre-order walk of the t-SNE solver plug-in (bh_forces with the t-SNE kernel, one system of
// at most kPreorderMax points). NBodySolver::solveNbody adds these sums to the caller's doubles,
// and they are kept bit for bit what they have been: their summation order is a wave's pre-order
// visits (128 sinks, monopoles folded every 8 visits and at every particle-particle cell), which
// k_walk's steps do not follow. The wave visits one node at a time; the records of both possible
// next visits are fetched with scalar loads while the current one is used; lanes that open a
// cell that others accept are pushed on a small LDS stack as lane masks.
// Bound by the latency of the visits: 20,011 points 0.21 ms (k_walk 0.09 ms).
// ------------------------------------------------------------------------------------------
constexpr int kPreNS = 2;  // sinks per lane
template <bool TOT>
__global__ __launch_bounds__(kBlock) void k_walk_preorder(const float4* __restrict__ pos4,
                                                          const Node* __restrict__ nodes,
                                                          const BuildParams* __restrict__ prm,
                                                          uint32_t n, float inv_theta2,
                                                          float* __restrict__ ax_out,
                                                          float* __restrict__ ay_out,
                                                          float* __restrict__ tot_out,
                                                          unsigned long long* __restrict__ counters) {
    constexpr int NS = kPreNS;
    __shared__ uint64_t st_mask[kWavesPerBlock][kStackDepth][NS];
    __shared__ uint32_t st_end[kWavesPerBlock][kStackDepth];
    const int lane = threadIdx.x & 63;
    // wave-uniform (the compiler cannot tell that threadIdx.x / 64 is): keeps the stack pointer,
    // the stack reads and the loop control in scalar registers
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wb = blockIdx.x;
    const uint32_t base = (wb * kWavesPerBlock + w) * (uint32_t)(kWave * NS);
    uint32_t idx[NS];
    bool valid[NS];
    float px[NS], py[NS], pm[NS];  // pm: the sink's own mass
    uint64_t active[NS];
    uint64_t any = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        idx[s] = base + s * kWave + lane;
        valid[s] = idx[s] < n;
        const float4 me = valid[s] ? pos4[idx[s]] : make_float4(0.f, 0.f, 0.f, 0.f);
        px[s] = me.x;
        pm[s] = me.z;
        py[s] = me.y;
        active[s] = __ballot(valid[s]);
        any |= active[s];
    }
    const uint32_t nn = prm->n_nodes;
    float ax[NS], ay[NS], at[NS], cax[NS], cay[NS], cat[NS], bx[NS], by[NS], bt[NS];
    uint32_t npn[NS], npp[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        ax[s] = ay[s] = at[s] = cax[s] = cay[s] = cat[s] = bx[s] = by[s] = bt[s] = 0.f;
        npn[s] = npp[s] = 0u;
    }
    uint32_t k = 0, end_cur = nn;
    int sp = 0, since_fold = 0;
    Node cur = nodes[min(0u, nn - 1)];
    while (any) {
        while (k == end_cur && sp > 0) {
            --sp;
#pragma unroll
            for (int s = 0; s < NS; ++s) active[s] = st_mask[w][sp][s];
            end_cur = st_end[w][sp];
        }
        if (k >= end_cur) break;
        // skip > k for every node of a well-formed tree; max() keeps the walk finite regardless
        const uint32_t next = max(cur.skip, k + 1);
        // the next node is k+1 (descend) or `next` (skip): fetch both while this one is used
        const Node nd_down = nodes[min(k + 1, nn - 1)];
        const Node nd_skip = nodes[min(next, nn - 1)];
        const float lim = cur.l2 * inv_theta2;
        uint64_t open[NS];
        uint64_t open_any = 0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const float dx = cur.cx - px[s], dy = cur.cy - py[s];
            const float d2 = fmaf(dx, dx, dy * dy);
            const bool on = (active[s] >> lane) & 1ull;
            const bool acc = on && (d2 > lim);
            if (__ballot(acc)) {
                const float wq = __builtin_amdgcn_rcpf(1.0f + d2);
                const float mw = cur.mass * wq;
                float f = mw * wq;
                f = acc ? f : 0.f;
                bx[s] = fmaf(-f, dx, bx[s]);
                by[s] = fmaf(-f, dy, by[s]);
                if (TOT) bt[s] += acc ? mw : 0.f;
                npn[s] += acc ? 1u : 0u;
            }
            open[s] = __ballot(on && !acc);
            open_any |= open[s];
        }
        bool down = false;
        if (open_any) {
            if (cur.meta & kMetaPP) {
                // every lane sums every source; lanes that did not open the cell drop the sums,
                // and the sink's own m * 1 is taken out of Z again
                bool mine[NS];
                float lx[NS], ly[NS], lt[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    mine[s] = ((open[s] >> lane) & 1ull) != 0ull;
                    lx[s] = ly[s] = lt[s] = 0.f;
                }
                const uint32_t f = cur.first, e = f + cur.count;
                auto pp_slots = [&](auto lo_c, auto hi_c) {
                    constexpr int LO = decltype(lo_c)::value, HI = decltype(hi_c)::value;
                    for (uint32_t j = f; j < e; ++j) {
                        const float4 q = pos4[j];
#pragma unroll
                        for (int s = LO; s < HI; ++s) {
                            const float qx = q.x - px[s], qy = q.y - py[s];
                            const float q2 = fmaf(qx, qx, qy * qy);
                            const float wq = __builtin_amdgcn_rcpf(1.0f + q2);
                            const float mw = q.z * wq;
                            const float sc = mw * wq;
                            lx[s] = fmaf(-sc, qx, lx[s]);
                            ly[s] = fmaf(-sc, qy, ly[s]);
                            if (TOT) lt[s] += mw;
                        }
                    }
                };
                using C0 = std::integral_constant<int, 0>;
                using C1 = std::integral_constant<int, 1>;
                using C2 = std::integral_constant<int, 2>;
                const bool a = open[0] != 0ull, c = open[1] != 0ull;
                if (a && c)
                    pp_slots(C0{}, C2{});
                else if (a)
                    pp_slots(C0{}, C1{});
                else if (c)
                    pp_slots(C1{}, C2{});
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    npp[s] += mine[s] ? (e - f) - ((idx[s] >= f && idx[s] < e) ? 1u : 0u) : 0u;
                    if (!mine[s]) lx[s] = ly[s] = lt[s] = 0.f;
                    if (TOT && mine[s] && idx[s] >= f && idx[s] < e) lt[s] -= pm[s];
                    kahan_add(ax[s], cax[s], lx[s] + bx[s]);
                    kahan_add(ay[s], cay[s], ly[s] + by[s]);
                    if (TOT) kahan_add(at[s], cat[s], lt[s] + bt[s]);
                    bx[s] = by[s] = bt[s] = 0.f;
                }
                since_fold = 0;
            } else {
                bool changed = false;
#pragma unroll
                for (int s = 0; s < NS; ++s) changed |= (open[s] != active[s]);
                if (changed && sp < kStackDepth) {
                    if (lane == 0) {
#pragma unroll
                        for (int s = 0; s < NS; ++s) st_mask[w][sp][s] = active[s];
                        st_end[w][sp] = end_cur;
                    }
                    ++sp;
#pragma unroll
                    for (int s = 0; s < NS; ++s) active[s] = open[s];
                    end_cur = next;
                }
                down = true;
            }
        }
        if (++since_fold >= kFoldEvery) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                kahan_add(ax[s], cax[s], bx[s]);
                kahan_add(ay[s], cay[s], by[s]);
                if (TOT) kahan_add(at[s], cat[s], bt[s]);
                bx[s] = by[s] = bt[s] = 0.f;
            }
            since_fold = 0;
        }
        k = down ? k + 1 : next;
        // select the next record word by word on the integer bit patterns: a uniform select
        // of uniform values, kept in scalar registers
        auto pick = [&](float a, float b) {
            return __uint_as_float(uniform_u32(down ? __float_as_uint(a) : __float_as_uint(b)));
        };
        cur.cx = pick(nd_down.cx, nd_skip.cx);
        cur.cy = pick(nd_down.cy, nd_skip.cy);
        cur.mass = pick(nd_down.mass, nd_skip.mass);
        cur.l2 = pick(nd_down.l2, nd_skip.l2);
        cur.skip = down ? nd_down.skip : nd_skip.skip;
        cur.first = down ? nd_down.first : nd_skip.first;
        cur.count = down ? nd_down.count : nd_skip.count;
        cur.meta = down ? nd_down.meta : nd_skip.meta;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        kahan_add(ax[s], cax[s], bx[s]);
        kahan_add(ay[s], cay[s], by[s]);
        if (TOT) kahan_add(at[s], cat[s], bt[s]);
        if (valid[s]) {
            ax_out[idx[s]] = ax[s] - cax[s];
            ay_out[idx[s]] = ay[s] - cay[s];
            if (TOT) tot_out[idx[s]] = at[s] - cat[s];
        }
    }
    unsigned long long s_pn = 0, s_pp = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        s_pn += valid[s] ? npn[s] : 0u;
        s_pp += valid[s] ? npp[s] : 0u;
    }
    s_pn = wave_sum_u64(s_pn);
    s_pp = wave_sum_u64(s_pp);
    if (lane == 0) {
        const size_t gw = (size_t)wb * kWavesPerBlock + w;
        counters[2 * gw] = s_pn;
        counters[2 * gw + 1] = s_pp;
    }
}

// ------------------------------------------------------------------------------------------
// FP64 reduction of per-particle totals (t-SNE Z, potential energy): fixed partition into
// block partials, then one block sums them in order, so the result is deterministic.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_reduce_f64_partial(const float* __restrict__ v,
                                                               uint32_t n,
                                                               const float* __restrict__ w,
                                                               double* __restrict__ partials) {
    double s = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        s += w ? (double)v[i] * (double)w[i] : (double)v[i];
    s = block_sum_d(s);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void k_reduce_f64_final(const double* __restrict__ partials,
                                                             uint32_t nb, double* __restrict__ out) {
    double s = 0.0;
    for (uint32_t b = threadIdx.x; b < nb; b += kBlock) s += partials[b];
    s = block_sum_d(s);
    if (threadIdx.x == 0) *out = s;
}

// Conserved quantities of the gravity state in FP64: per block the partial sums of kinetic
// energy sum m (vx^2 + vy^2) / 2, potential energy sum m phi / 2 (phi = the walk's per-particle
// potential, G included) and momentum sum m v; then one block adds the partials in block order.
__global__ __launch_bounds__(kBlock) void k_state_partial(const float* __restrict__ m,
                                                          const float* __restrict__ vx,
                                                          const float* __restrict__ vy,
                                                          const float* __restrict__ phi, uint32_t n,
                                                          double* __restrict__ partials) {
    double ke = 0.0, pe = 0.0, px = 0.0, py = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const double mi = m[i], u = vx[i], v = vy[i];
        ke += 0.5 * mi * (u * u + v * v);
        pe += 0.5 * mi * (double)phi[i];
        px += mi * u;
        py += mi * v;
    }
    ke = block_sum_d(ke);
    pe = block_sum_d(pe);
    px = block_sum_d(px);
    py = block_sum_d(py);
    if (threadIdx.x == 0) {
        partials[4 * (size_t)blockIdx.x + 0] = ke;
        partials[4 * (size_t)blockIdx.x + 1] = pe;
        partials[4 * (size_t)blockIdx.x + 2] = px;
        partials[4 * (size_t)blockIdx.x + 3] = py;
    }
}

__global__ __launch_bounds__(kBlock) void k_state_final(const double* __restrict__ partials,
                                                        uint32_t nb, double* __restrict__ out) {
    double r[4] = {0.0, 0.0, 0.0, 0.0};
    for (uint32_t b = threadIdx.x; b < nb; b += kBlock)
        for (int q = 0; q < 4; ++q) r[q] += partials[4 * (size_t)b + q];
    for (int q = 0; q < 4; ++q) {
        const double t = block_sum_d(r[q]);
        if (threadIdx.x == 0) out[q] = t;
    }
}

// out[id[i]] = a[i] (results back to the caller's particle order)
__global__ __launch_bounds__(kBlock) void k_unsort2(const uint32_t* __restrict__ id, uint32_t n,
                                                    const float* __restrict__ a,
                                                    const float* __restrict__ b,
                                                    float* __restrict__ ao, float* __restrict__ bo) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = id[i];
    ao[j] = a[i];
    if (b) bo[j] = b[i];
}

// unsorts a and b and sums w per block (partials in FP64)
__global__ __launch_bounds__(kBlock) void k_unsort2_sum(const uint32_t* __restrict__ id, uint32_t n,
                                                        const float* __restrict__ a,
                                                        const float* __restrict__ b,
                                                        const float* __restrict__ w,
                                                        float* __restrict__ ao,
                                                        float* __restrict__ bo,
                                                        double* __restrict__ partials) {
    double s = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const uint32_t j = id[i];
        ao[j] = a[i];
        bo[j] = b[i];
        s += (double)w[i];
    }
    s = block_sum_d(s);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// kick-drift of kick-drift-kick leapfrog, v += a dt/2; x += v dt, and the partial bounds of the new
// positions for the build that follows. close: the closing kick of the step before goes first (two
// kicks, rounded as two). One launch where three stood (kick, kick-drift, bounds: 14 -> 5 us at
// 200k particles).
__global__ __launch_bounds__(kBlock) void k_kick_drift(float* __restrict__ x, float* __restrict__ y,
                                                       float* __restrict__ vx,
                                                       float* __restrict__ vy,
                                                       const float* __restrict__ ax,
                                                       const float* __restrict__ ay, uint32_t n,
                                                       float hdt, float dt, int close,
                                                       float4* __restrict__ bounds) {
    float4 box = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const float a = ax[i], b = ay[i];
        float u = vx[i], v = vy[i];
        if (close) {
            u = fmaf(a, hdt, u);
            v = fmaf(b, hdt, v);
        }
        u = fmaf(a, hdt, u);
        v = fmaf(b, hdt, v);
        vx[i] = u;
        vy[i] = v;
        const float px = fmaf(u, dt, x[i]), py = fmaf(v, dt, y[i]);
        x[i] = px;
        y[i] = py;
        box = minmax4(box, bounds_item(px, py));
    }
    box = block_minmax4(box);
    if (threadIdx.x == 0) bounds[blockIdx.x] = box;
}

__global__ __launch_bounds__(kBlock) void k_kick(float* __restrict__ vx, float* __restrict__ vy,
                                                 const float* __restrict__ ax,
                                                 const float* __restrict__ ay, uint32_t n,
                                                 float hdt) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    vx[i] = fmaf(ax[i], hdt, vx[i]);
    vy[i] = fmaf(ay[i], hdt, vy[i]);
}

// ------------------------------------------------------------------------------------------
static inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// Waves per sink group, results do not depend on it. Measured with 1 / 2 / 4 waves:
//   uniform disk, 20,000 sinks (313 groups)    130 / 107 /  91 us
//   t-SNE, 70,000 points (1,094 groups)        162 / 139 / 141 us compact, 141 / 117 / 111 spread
//   two disks, 200,003 sinks (3,126 groups)    200 / 209 / 285 us; 1,048,576: 654 / 806 / 1215 us
// So four waves while the groups alone leave SIMDs idle, two up to two groups per SIMD. Around one
// group per SIMD (1,024), the time with four waves over the time with two, theta 0.4 to 1.1 on two
// disks, a uniform and a Plummer disk (t-SNE: spread and compact):
//   groups            969         1,025-1,047  1,079-1,110  1,152       1,204       1,563
//   gravity           0.93-1.02   0.95-1.02    0.96-1.06    0.98-1.08   0.98-1.04   1.15-1.26
//   with the total    0.92-1.01   0.92-1.02    0.95-1.06    0.95-1.06   0.95-1.02   1.09-1.12
//   learned           0.95        0.85-0.92    0.87-0.95    0.90-0.95   0.91-0.95   0.92-1.09
//   t-SNE             0.72-0.97   0.83-0.98    0.68-0.95    0.79-0.95   0.66-0.98   0.80-1.08
// Gravity is even there (the smaller angles gain what the larger ones lose), the learned walk and
// t-SNE gain (beside the attraction 1470 -> 1448 us for five iterations, compact, 1500 -> 1475
// spread): four waves for an eighth of a group per SIMD more.
static uint64_t walk_simds() {
    static const uint64_t simds = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            cus = 0;
        return (uint64_t)cus * 4u;
    }();
    return simds;
}

static uint32_t walk_waves_per_group(uint64_t groups) {
    const uint64_t simds = walk_simds();
    return groups <= simds + simds / 8 ? 4u : groups <= 2 * simds ? 2u : 1u;
}

// One wave per group: left to itself the compiler takes 88 to 106 registers, five (with totals four)
// waves per SIMD. Launches that bring more groups than that run a build held to the
// registers of six or seven resident waves: a few values go through scratch, and the added waves
// hide the loads and LDS reads. Where fewer groups come, the spills cost and nothing is gained.
// Compiler's own / six / seven / eight, theta 0.5, us:
//   two disks,   200,000 sinks  217 /  221 /  232 /  283      with totals  237 /  261 /  357
//              1,048,576        663 /  627 /  635 /  746                   790 /  728 / 1000
//              4,194,304       2381 / 2212 / 2195 / 2634
//   t-SNE,       400,000        284 /  265 /  248 /  263                   321 /  314 /  293
//   64 systems (2.9M sinks)    1242 / 1156 / 1099 / 1675                  1511 / 1344 / 1870
//   learned,   4,194,304       2636 / 2524 / 2522 / 2735
constexpr uint64_t kWalkResident = 5;
static constexpr int walk_resident(int kernel, bool tot, bool batched) {
    return kernel == kKernelTsne || (batched && !tot) ? 7 : 6;
}

struct WalkCall {
    hipStream_t s;
    const float4* pos4;
    const Node* nodes;
    const uint32_t* child4;
    const BuildParams* prm;
    uint32_t n;
    float inv_theta2, eps2, scale;
    float *ax, *ay, *tot;
    unsigned long long* counters;
    TraverseBatch batch;
    LearnArgs la;
    uint32_t waves;  // per sink group: 1, 2 or 4
    CallerOut out;
};

template <int KERNEL, bool TOT, bool BATCHED, int LTERMS>
static uint32_t walk_launch(const WalkCall& c) {
    const uint64_t groups = BATCHED ? c.batch.n_work : div_up(c.n, kWave);
    const uint32_t g = div_up(groups * c.waves, kWavesPerBlock);
#define BH_WALK(NP, RES)                                                                          \
    k_walk<KERNEL, TOT, NP, BATCHED, LTERMS, RES><<<g, kBlock, 0, c.s>>>(                         \
        c.pos4, c.nodes, c.child4, c.prm, c.n, c.inv_theta2, c.eps2, c.scale, c.ax, c.ay, c.tot,  \
        c.counters, c.batch, c.la, c.out)
    if (c.waves == 4) BH_WALK(1, 1);
    else if (c.waves == 2) BH_WALK(2, 1);
    else if (groups <= kWalkResident * walk_simds()) BH_WALK(4, 1);
    else BH_WALK(4, walk_resident(KERNEL, TOT, BATCHED));
#undef BH_WALK
    return g;
}

uint32_t launch_traverse(hipStream_t s, int kernel, const float4* pos4, const Node* nodes,
                         const uint32_t* child4, const BuildParams* prm, uint32_t n,
                         float inv_theta2, float eps2, float scale, float* ax, float* ay,
                         float* tot, unsigned long long* counters, TraverseBatch batch,
                         uint32_t split, CallerOut out) {
    WalkCall c{s, pos4, nodes, child4, prm, n, inv_theta2, eps2, scale, ax, ay, tot, counters,
               batch, LearnArgs{}, 1u, out};
    if (split > 1) c.waves = split == 2 ? 2u : 4u;
    else if (!batch.work) c.waves = walk_waves_per_group(div_up(n, kWave));
    const bool grav = kernel == kKernelGravity;
    if (batch.work) {
        if (grav) return tot ? walk_launch<kKernelGravity, true, true, 0>(c)
                             : walk_launch<kKernelGravity, false, true, 0>(c);
        return tot ? walk_launch<kKernelTsne, true, true, 0>(c)
                   : walk_launch<kKernelTsne, false, true, 0>(c);
    }
    if (grav) return tot ? walk_launch<kKernelGravity, true, false, 0>(c)
                         : walk_launch<kKernelGravity, false, false, 0>(c);
    return tot ? walk_launch<kKernelTsne, true, false, 0>(c)
               : walk_launch<kKernelTsne, false, false, 0>(c);
}

uint32_t launch_traverse_preorder(hipStream_t s, const float4* pos4, const Node* nodes,
                                  const BuildParams* prm, uint32_t n, float inv_theta2, float* ax,
                                  float* ay, float* tot, unsigned long long* counters) {
    const uint32_t g = div_up(n, kBlock * kPreNS);
    if (tot)
        k_walk_preorder<true><<<g, kBlock, 0, s>>>(pos4, nodes, prm, n, inv_theta2, ax, ay, tot,
                                                   counters);
    else
        k_walk_preorder<false><<<g, kBlock, 0, s>>>(pos4, nodes, prm, n, inv_theta2, ax, ay, tot,
                                                    counters);
    return g;
}

uint32_t launch_traverse_learned(hipStream_t s, const float4* pos4, const Node* nodes,
                                 const uint32_t* child4, const float4* coef,
                                 const BuildParams* prm, uint32_t n, float inv_theta2,
                                 float inv_band2, float eps2, float scale, int terms, float* ax,
                                 float* ay, float* tot, unsigned long long* counters,
                                 CallerOut out) {
    WalkCall c{s, pos4, nodes, child4, prm, n, inv_theta2, eps2, scale, ax, ay, tot, counters,
               TraverseBatch{}, LearnArgs{coef, inv_band2}, walk_waves_per_group(div_up(n, kWave)), out};
    if (terms == 3)
        return tot ? walk_launch<kKernelGravity, true, false, 3>(c)
                   : walk_launch<kKernelGravity, false, false, 3>(c);
    return tot ? walk_launch<kKernelGravity, true, false, 7>(c)
               : walk_launch<kKernelGravity, false, false, 7>(c);
}

// heavy batched entries: out[first + i] = sum over slices f of side[slot][f][i], in slice order
// (one block per slot)
__global__ __launch_bounds__(kBlock) void k_sum_heavy(const float* __restrict__ side,
                                                      uint32_t side_slots,
                                                      const uint4* __restrict__ heavy,
                                                      float* __restrict__ ax,
                                                      float* __restrict__ ay,
                                                      float* __restrict__ tot, CallerOut out) {
    const uint4 h = heavy[blockIdx.x];  // first sink, count, F
    const size_t plane = (size_t)side_slots * kHeavySlices * kHeavySinks;
    for (uint32_t i = threadIdx.x; i < h.y; i += kBlock) {
        float sx = 0.f, sy = 0.f, st = 0.f;
        for (uint32_t f = 0; f < h.z; ++f) {
            const size_t o = ((size_t)blockIdx.x * kHeavySlices + f) * kHeavySinks + i;
            sx += side[o];
            sy += side[plane + o];
            if (tot) st += side[2 * plane + o];
        }
        ax[h.x + i] = sx;
        ay[h.x + i] = sy;
        if (tot) tot[h.x + i] = st;
        if (out.id) {
            const uint32_t o = out.id[h.x + i];
            if (out.x) out.x[o] = sx;
            if (out.y) out.y[o] = sy;
        }
    }
}

void launch_sum_heavy(hipStream_t s, const float* side, uint32_t side_slots, const uint4* heavy,
                      uint32_t nheavy, float* ax, float* ay, float* tot, CallerOut out) {
    if (nheavy) k_sum_heavy<<<nheavy, kBlock, 0, s>>>(side, side_slots, heavy, ax, ay, tot, out);
}

uint32_t reduce_grid(uint32_t n) {
    uint32_t g = div_up(n, kBlock * 16);
    if (g < 1) g = 1;
    if (g > kMaxReduceBlocks) g = kMaxReduceBlocks;
    return g;
}

void launch_state_sums(hipStream_t s, const float* m, const float* vx, const float* vy,
                       const float* phi, uint32_t n, double* partials, double* out) {
    const uint32_t g = reduce_grid(n) < kMaxReduceBlocks / 4 ? reduce_grid(n) : kMaxReduceBlocks / 4;
    k_state_partial<<<g, kBlock, 0, s>>>(m, vx, vy, phi, n, partials);
    k_state_final<<<1, kBlock, 0, s>>>(partials, g, out);
}

void launch_reduce_f64(hipStream_t s, const float* v, const float* w, uint32_t n, double* partials,
                       double* out) {
    const uint32_t g = reduce_grid(n);
    k_reduce_f64_partial<<<g, kBlock, 0, s>>>(v, n, w, partials);
    k_reduce_f64_final<<<1, kBlock, 0, s>>>(partials, g, out);
}

uint32_t traverse_blocks(uint32_t n) { return div_up(n, kBlock); }

void launch_unsort2(hipStream_t s, const uint32_t* id, uint32_t n, const float* a, const float* b,
                    float* ao, float* bo) {
    k_unsort2<<<div_up(n, kBlock), kBlock, 0, s>>>(id, n, a, b, ao, bo);
}

uint32_t launch_unsort2_sum(hipStream_t s, const uint32_t* id, uint32_t n, const float* a,
                            const float* b, const float* w, float* ao, float* bo,
                            double* partials) {
    const uint32_t g = min(div_up(n, kBlock), kMaxReduceBlocks);
    k_unsort2_sum<<<g, kBlock, 0, s>>>(id, n, a, b, w, ao, bo, partials);
    return g;
}

uint32_t update_blocks(uint32_t n) { return min(div_up(n, kBlock), kMaxBoundsBlocks); }

void launch_kick_drift(hipStream_t s, float* x, float* y, float* vx, float* vy, const float* ax,
                       const float* ay, uint32_t n, float hdt, float dt, bool close,
                       float4* bounds) {
    k_kick_drift<<<update_blocks(n), kBlock, 0, s>>>(x, y, vx, vy, ax, ay, n, hdt, dt, close ? 1 : 0,
                                                     bounds);
}

void launch_kick(hipStream_t s, float* vx, float* vy, const float* ax, const float* ay, uint32_t n,
                 float hdt) {
    k_kick<<<div_up(n, kBlock), kBlock, 0, s>>>(vx, vy, ax, ay, n, hdt);
}

}  // namespace bh
