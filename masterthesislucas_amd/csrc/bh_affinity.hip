// t-SNE input affinities on gfx950: exact k nearest neighbours, a Gaussian bandwidth per point
// found by bisection to a perplexity, and the symmetrised sparse P = (P_cond + P_cond^T) / (2n)
// in CSR sorted by (row, column).
//
// The reference prepares P offline (MnistLoader.ipynb:539-547, openTSNE's exact
// PerplexityBasedNN and joint_probabilities_nn) and loads it from a Matrix Market file
// (tsne.h:94-98); setupEfficientPmatrix keeps it as row-sorted CSR (tsne.h:462-520).
//
// Neighbours. Candidates come from FP16 Gram products on MFMA (v_mfma_f32_16x16x32_f16, FP32
// accumulation), exact ones from FP64 distances of the FP32 inputs. Each (i, j) gets rigorous
// bounds [lo, hi] of the exact Euclidean distance: with x^ the FP16 rounding of the scaled
// point x (|x - x^| <= 2^-11 |x| + sqrt(dim) 2^-25, scaled units, RNE with subnormals) and d^
// the FP32 value of |x^_i|^2 + |x^_j|^2 - 2 x^_i.x^_j (error at most
// delta = 2^-24 ((2K + 4) |x^_i| |x^_j| + 4 (|x^_i|^2 + |x^_j|^2)) for K accumulated products),
// |x_i - x_j| lies in [sqrt(d^ - delta) - e_i - e_j, sqrt(d^ + delta) + e_i + e_j]. A row keeps
// every column whose lower bound does not exceed T, the k-th smallest upper bound seen so far,
// so the final candidates contain the exact k nearest; their FP64 distances decide, ties by
// index. A row whose candidate window outgrows its buffer is reported (an error, never a
// silently wrong neighbour list).
#include "bh_common.h"
#include "bh_launch.h"

namespace bh {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ static inline uint32_t div_up_a(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

constexpr int kAffRows = 128;                 // query rows per workgroup
constexpr int kAffCols = 256;                 // candidate columns per tile
constexpr int kAffKC = 64;                    // K halfs per staged chunk
constexpr int kAffPad = 8;                    // LDS row padding (bank spread of 16-byte reads)
constexpr uint32_t kAffCap = 512;             // candidate slots per row and column range
constexpr uint32_t kAffHold = kAffCap - kAffCols;  // compact above this many (a tile adds <= 256)
constexpr uint32_t kAffKeep = 192;            // most candidates of a row over all columns
constexpr uint32_t kAffMaxSplits = 4;         // most column ranges
constexpr uint32_t kAffOver = 1u << 31;       // flag of a list's count: its window outgrew the buffer

// largest magnitude bits of the inputs (order = |x|; infinities and NaN above every finite one),
// into *out (cleared by the caller); one integer atomic per block
__global__ __launch_bounds__(kBlock) void k_aff_maxbits(const uint32_t* __restrict__ x, uint64_t n,
                                                        uint32_t* __restrict__ out) {
    __shared__ uint32_t red[kWavesPerBlock];
    uint32_t m = 0;
    for (uint64_t e = (uint64_t)blockIdx.x * kBlock + threadIdx.x; e < n;
         e += (uint64_t)gridDim.x * kBlock)
        m = max(m, x[e] & 0x7FFFFFFFu);
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, kWave));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kWavesPerBlock; ++w) m = max(m, red[w]);
        atomicMax(out, m);
    }
}

// ---------------------------------------------------------------------------------------------
// scaled FP16 copy, squared norms and rounding bounds (one wave per point)
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_aff_pack(const float* __restrict__ X, uint32_t n,
                                                     uint32_t dim, uint32_t dp, float2 scale,
                                                     _Float16* __restrict__ Xh,
                                                     float* __restrict__ nh,
                                                     float* __restrict__ ah,
                                                     float* __restrict__ eb) {
    const int lane = threadIdx.x & 63;
    const uint32_t i = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (i >= n) return;
    double sh = 0.0, sx = 0.0;
    for (uint32_t e = lane; e < dp; e += kWave) {
        // 2^m in two factors: for the smallest inputs m exceeds a float's exponent
        const float v = e < dim ? X[(size_t)i * dim + e] * scale.x * scale.y : 0.f;
        const _Float16 h = (_Float16)v;
        Xh[(size_t)i * dp + e] = h;
        const double hd = (double)h;
        sh += hd * hd;
        sx += (double)v * (double)v;
    }
    sh = wave_sum_d(sh);
    sx = wave_sum_d(sx);
    if (lane == 0) {
        nh[i] = (float)sh;
        ah[i] = (float)sqrt(sh) * (1.0f + 0x1p-20f);
        eb[i] = (float)(0x1p-11 * sqrt(sx) + sqrt((double)dim) * 0x1p-25) * (1.0f + 0x1p-20f);
    }
}

// ---------------------------------------------------------------------------------------------
// candidates: a workgroup owns kAffRows query rows and streams the columns of its range in tiles
// of kAffCols; the range is all columns, or one of `splits` equal ranges where the row blocks
// alone leave compute units idle (k_aff_refine merges a row's lists)
// ---------------------------------------------------------------------------------------------
// one wave, PER entries per lane: a bit pattern t with #(hb <= t among valid) >= k, found in at
// most `steps` halvings of the range of the entries; 32 steps give the smallest one (upper bounds
// are >= 0, so their bits order them). At least k entries are valid.
template <int PER>
__device__ __forceinline__ uint32_t aff_kth(const uint32_t (&hb)[PER], const bool (&v)[PER],
                                            uint32_t k, int steps) {
    uint32_t a = 0xFFFFFFFFu, b = 0u;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        a = min(a, v[u] ? hb[u] : 0xFFFFFFFFu);
        b = max(b, v[u] ? hb[u] : 0u);
    }
    for (int o = 32; o > 0; o >>= 1) {
        a = min(a, (uint32_t)__shfl_xor((int)a, o, kWave));
        b = max(b, (uint32_t)__shfl_xor((int)b, o, kWave));
    }
    a = (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
    b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
    for (int it = 0; it < steps && a < b; ++it) {
        const uint32_t mid = a + ((b - a) >> 1);
        uint32_t m = 0;
#pragma unroll
        for (int u = 0; u < PER; ++u) m += (uint32_t)__popcll(__ballot(v[u] && hb[u] <= mid));
        if (m >= k) b = mid; else a = mid + 1;
    }
    return b;
}

// Bounds [lo, hi] of the exact distance of a pair from its Gram value g (header comment):
// ni, ai, ei and nj, aj, ej are |x^|^2, |x^| (rounded up) and the rounding bound of its points.
__device__ __forceinline__ void aff_bounds(float g, float kdelta, float ni, float ai, float ei,
                                           float nj, float aj, float ej, float& lo, float& hi) {
    const float sn = ni + nj, d = sn - 2.0f * g;
    const float delta = (kdelta * ai * aj + 0x1p-22f * sn) * (1.0f + 0x1p-20f);
    const float e2 = (ei + ej) * (1.0f + 0x1p-20f);
    lo = sqrtf(fmaxf(d - delta, 0.f)) * (1.0f - 0x1p-20f) - e2;
    lo -= fabsf(lo) * 0x1p-22f;
    hi = (sqrtf(fmaxf(d + delta, 0.f)) * (1.0f + 0x1p-20f) + e2) * (1.0f + 0x1p-22f);
}

// Per point |x^|^2, |x^| and the rounding bound (k_aff_pack)
struct AffPoints {
    const float *nh, *ah, *eb;
};
__device__ __forceinline__ float aff_kdelta(uint32_t dp) { return 0x1p-24f * (float)(2 * dp + 4); }

// Compact row i's candidate list (one wave), its entries (column, Gram value) already in `en`:
// T = min(T, about the k-th smallest upper bound), keep the entries whose lower bound is at most
// T, in order. T comes from ten halvings (a wave needs no more to thin the list); a window that
// does not fit is settled with the exact k-th.
constexpr int kAffPer = kAffCap / kWave;
__device__ __forceinline__ void aff_load(const uint2* __restrict__ list, uint32_t c, uint32_t i,
                                         uint2 (&en)[kAffPer]) {
#pragma unroll
    for (int u = 0; u < kAffPer; ++u) {
        const uint32_t q = (threadIdx.x & 63) + 64u * u;
        en[u] = q < c ? list[q] : make_uint2(i, 0u);
    }
}
__device__ __forceinline__ void aff_compact(uint2* __restrict__ list, AffPoints P, uint32_t dp,
                                            uint32_t i, const uint2 (&en)[kAffPer], uint32_t* cnt,
                                            float* T, uint32_t* over, uint32_t k) {
    const int lane = threadIdx.x & 63;
    const uint32_t c = *cnt;
    const float kd = aff_kdelta(dp), ni = P.nh[i], ai = P.ah[i], ei = P.eb[i];
    uint32_t hb[kAffPer];
    float lo[kAffPer];
    bool v[kAffPer];
#pragma unroll
    for (int u = 0; u < kAffPer; ++u) {
        v[u] = lane + 64u * u < c;
        float hi;
        aff_bounds(__uint_as_float(en[u].y), kd, ni, ai, ei, P.nh[en[u].x], P.ah[en[u].x],
                   P.eb[en[u].x], lo[u], hi);
        hb[u] = __float_as_uint(hi);
    }
    const float t0 = *T;
    float t = t0;
    uint32_t base = 0;
    uint64_t keep[kAffPer];
    for (int steps = 10;; steps = 32) {
        if (c >= k) t = fminf(t0, __uint_as_float(aff_kth<kAffPer>(hb, v, k, steps)));
        base = 0;
#pragma unroll
        for (int u = 0; u < kAffPer; ++u) {
            keep[u] = __ballot(v[u] && lo[u] <= t);
            base += (uint32_t)__popcll(keep[u]);
        }
        if (base <= kAffHold || steps == 32) break;
    }
    uint32_t at = 0;
#pragma unroll
    for (int u = 0; u < kAffPer; ++u) {
        const uint32_t pos = at + (uint32_t)__popcll(keep[u] & lane_mask_lt());
        if (((keep[u] >> lane) & 1ull) && pos < kAffHold) list[pos] = en[u];
        at += (uint32_t)__popcll(keep[u]);
    }
    if (lane == 0) {
        *T = t;
        if (base > kAffHold) *over = 1u;  // the window outgrew the buffer: reported, not used
        *cnt = min(base, kAffHold);
    }
}

// lane 0 of each row of 16 lanes to the whole row (DPP row_newbcast:0)
__device__ __forceinline__ uint32_t row_first(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150, 0xF, 0xF, false);
}

// the threshold of a row as the other column ranges' workgroups have it so far (any of them bounds
// the k-th smallest distance over all columns; upper bounds are >= 0, so their bits order them)
__device__ __forceinline__ float aff_thr(const uint32_t* p) {
    return __uint_as_float(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Workgroup: 8 waves as 2 x 4 over a 128 x 256 tile of Gram products, 64 x 64 per wave (16
// v_mfma_f32_16x16x32_f16 tiles from 4 + 4 operand reads per K step of 32). Rows and columns
// stream through LDS in chunks of 64 halfs, double-buffered: the next chunk's global loads are
// in flight while the current one feeds the MFMAs. Bound by the matrix cores and the LDS reads
// that feed them (8 reads of 1 KB per 16 MFMAs; the earlier 16 x 64 tile per wave read LDS once
// per MFMA and left the matrix cores three quarters idle). The epilogue tests every pair with one
// addition and comparison, then the few that pass against the row's threshold without square
// roots, conservatively, and appends (column, Gram value); the bounds themselves are taken when a
// row's list is compacted, 64 entries at a time. Workgroups of the same rows share their
// thresholds: those that start later collect a fraction of the candidates. 20,000 points in 784-D:
// 4.68 ms with 16 x 64 products per wave, 2.49 with 64 x 64, 1.87 with the short test and the
// shared thresholds.
constexpr int kAffThreads = 512;
constexpr int kAffLd = kAffKC + kAffPad;
constexpr int kAffLoads = (kAffRows + kAffCols) * (kAffKC / 8) / kAffThreads;  // 16 B per thread
static_assert(kAffLoads * kAffThreads == (kAffRows + kAffCols) * (kAffKC / 8), "chunk loads");

__global__ __launch_bounds__(kAffThreads) void k_aff_candidates(const _Float16* __restrict__ Xh,
                                                                const float* __restrict__ nh,
                                                                const float* __restrict__ ah,
                                                                const float* __restrict__ eb,
                                                                uint32_t n, uint32_t dp,
                                                                uint32_t k,
                                                                uint2* __restrict__ cand,
                                                                uint32_t* __restrict__ ccount,
                                                                uint32_t* thr) {
    __shared__ __attribute__((aligned(16))) _Float16 s_t[2][(kAffRows + kAffCols) * kAffLd];
    __shared__ uint32_t s_cnt[kAffRows], s_over[kAffRows];
    __shared__ float s_T[kAffRows], s_nh[kAffRows], s_ka[kAffRows], s_eb[kAffRows];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = w >> 2, wc = w & 3;
    const int r16 = lane & 15, q4 = lane >> 4;
    const uint32_t row0 = blockIdx.x * kAffRows;
    const uint32_t ntiles = div_up_a(n, kAffCols);
    const uint32_t t0 = (uint32_t)((uint64_t)ntiles * blockIdx.y / gridDim.y);
    const uint32_t t1 = (uint32_t)((uint64_t)ntiles * (blockIdx.y + 1) / gridDim.y);
    const size_t lists = (size_t)blockIdx.y * n;  // this column range's lists: row i at lists + i
    const AffPoints P{nh, ah, eb};
    // the test's factors: delta's and the threshold's a little larger than aff_bounds takes them
    constexpr float kUp = 1.0f + 0x1p-17f;
    if (tid < kAffRows) {
        const uint32_t i = row0 + tid;
        s_cnt[tid] = 0u;
        s_over[tid] = 0u;
        s_T[tid] = i < n ? aff_thr(thr + i) : INFINITY;
        s_nh[tid] = i < n ? nh[i] : 0.f;
        s_ka[tid] = i < n ? aff_kdelta(dp) * ah[i] * kUp : 0.f;
        s_eb[tid] = i < n ? eb[i] * kUp : 0.f;
    }
    const uint32_t nch = dp / kAffKC, nchunks = (t1 - t0) * nch;  // (tile, K chunk) in order
    half8 pre[kAffLoads];
    auto fetch = [&](uint32_t tile, uint32_t ch) {
#pragma unroll
        for (int u = 0; u < kAffLoads; ++u) {
            const int e = tid + u * kAffThreads;
            const int q = e & (kAffKC / 8 - 1), rc = e / (kAffKC / 8);
            const uint32_t g = rc < kAffRows ? row0 + rc : tile * kAffCols + (rc - kAffRows);
            pre[u] = g < n ? *(const half8*)(Xh + (size_t)g * dp + ch * kAffKC + q * 8) : half8{};
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int u = 0; u < kAffLoads; ++u) {
            const int e = tid + u * kAffThreads;
            const int q = e & (kAffKC / 8 - 1), rc = e / (kAffKC / 8);
            *(half8*)(&s_t[buf][rc * kAffLd + q * 8]) = pre[u];
        }
    };
    if (nchunks) {
        fetch(t0, 0);
        stage(0);
    }
    __syncthreads();
    uint32_t c = 0;
    for (uint32_t t = t0; t < t1; ++t) {
        // the epilogue's column constants, in flight during the products
        const uint32_t c0 = t * kAffCols;
        f32x4 nj, aj, ej;
        bool jv[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const uint32_t j = c0 + 64 * wc + 16 * b + r16;
            jv[b] = j < n;
            nj[b] = jv[b] ? nh[j] : 0.f;
            aj[b] = jv[b] ? ah[j] : 0.f;
            ej[b] = jv[b] ? eb[j] * kUp : 0.f;
        }
        const float theirs = tid < kAffRows && row0 + tid < n ? aff_thr(thr + row0 + tid) : INFINITY;
        f32x4 acc[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t ch = 0; ch < nch; ++ch, ++c) {
            const int buf = c & 1;
            const bool more = c + 1 < nchunks;
            if (more) fetch(ch + 1 < nch ? t : t + 1, ch + 1 < nch ? ch + 1 : 0);
            const _Float16* A = &s_t[buf][(64 * wr + r16) * kAffLd + 8 * q4];
            const _Float16* Bp = &s_t[buf][(kAffRows + 64 * wc + r16) * kAffLd + 8 * q4];
#pragma unroll
            for (int s = 0; s < kAffKC / 32; ++s) {
                half8 av[4], bv[4];
#pragma unroll
                for (int a = 0; a < 4; ++a) av[a] = *(const half8*)(A + 16 * a * kAffLd + 32 * s);
#pragma unroll
                for (int b = 0; b < 4; ++b) bv[b] = *(const half8*)(Bp + 16 * b * kAffLd + 32 * s);
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[a], bv[b], acc[a][b],
                                                                           0, 0, 0);
            }
            // the other buffer was last read in the previous chunk, before its barrier
            if (more) stage(buf ^ 1);
            __syncthreads();
        }
        // acc[a][b][e] = x^_i . x^_j, i = row0 + 64 wr + 16 a + 4 q4 + e, j = c0 + 64 wc + 16 b + r16.
        // A pair that passes the threshold test has g >= (its row's term) + (its column's), the
        // terms with the largest |x^_j| and rounding bound of the wave's columns and a slack of
        // 2^-19 |x^|^2 over their own rounding: one addition and one comparison per pair.
        const bool edge = c0 < row0 + kAffRows && row0 < c0 + kAffCols;  // holds pairs with j = i
        float am = 0.f, em = 0.f, hc[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            am = fmaxf(am, aj[b]);
            em = fmaxf(em, ej[b]);
            hc[b] = jv[b] ? 0.5f * nj[b] * (1.0f - 0x1p-19f) : INFINITY;
        }
        for (int o = 8; o > 0; o >>= 1) {  // over the 16 columns of a row of lanes
            am = fmaxf(am, __shfl_xor(am, o, kWave));
            em = fmaxf(em, __shfl_xor(em, o, kWave));
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            uint32_t hits = 0;  // bit 4 e + b
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int il = 64 * wr + 16 * a + 4 * q4 + e;
                const float te = fmaf(s_T[il], kUp, s_eb[il]) + em;
                const float hr = row0 + il < n
                                     ? 0.5f * fmaf(-te * (1.0f + 0x1p-19f), te,
                                                   s_nh[il] * (1.0f - 0x1p-19f) - s_ka[il] * am * kUp)
                                     : INFINITY;
#pragma unroll
                for (int b = 0; b < 4; ++b) hits |= acc[a][b][e] >= hr + hc[b] ? 1u << (4 * e + b) : 0u;
            }
            // a lane's few hits, tested as the bounds have them and appended one at a time
            while (hits) {
                const uint32_t x = (uint32_t)__builtin_ctz(hits);
                hits &= hits - 1;
                const uint32_t e = x >> 2, b = x & 3u;
                auto pick = [](f32x4 c, uint32_t x) {  // no memory: selects
                    const float p = x & 1u ? c[1] : c[0], q = x & 1u ? c[3] : c[2];
                    return x & 2u ? q : p;
                };
                const f32x4 v = {pick(acc[a][0], e), pick(acc[a][1], e), pick(acc[a][2], e),
                                 pick(acc[a][3], e)};
                const float gv = pick(v, b);
                const uint32_t il = 64 * wr + 16 * a + 4 * q4 + e;
                const uint32_t i = row0 + il, j = c0 + 64 * wc + 16 * b + r16;
                const float sn = s_nh[il] + pick(nj, b);
                const float te = fmaf(s_T[il], kUp, s_eb[il]) + pick(ej, b);
                const float dm = fmaf(-s_ka[il], pick(aj, b), fmaf(-0x1p-21f, sn, sn - 2.0f * gv));
                if (dm > te * te || (edge && j == i)) continue;
                const uint32_t at = atomicAdd(&s_cnt[il], 1u);  // < kAffCap: at most kAffHold before
                cand[(lists + i) * kAffCap + at] = make_uint2(j, __float_as_uint(gv));
            }
        }
        __syncthreads();
        // rows whose buffer could overflow with the next tile are compacted, a wave per row
        uint64_t need = __ballot(lane < kAffRows / 8 && s_cnt[w * (kAffRows / 8) + (lane & 15)] > kAffHold);
        uint2 en[kAffPer], nx[kAffPer];
        int r = w * (kAffRows / 8) + (need ? __builtin_ctzll(need) : 0);
        if (need) aff_load(cand + (lists + row0 + r) * kAffCap, s_cnt[r], row0 + r, en);
        while (need) {
            need &= need - 1;
            const int rn = w * (kAffRows / 8) + (need ? __builtin_ctzll(need) : 0);
            if (need)  // the next row's entries are in flight during this row's selection
                aff_load(cand + (lists + row0 + rn) * kAffCap, s_cnt[rn], row0 + rn, nx);
            aff_compact(cand + (lists + row0 + r) * kAffCap, P, dp, row0 + r, en, &s_cnt[r],
                        &s_T[r], &s_over[r], k);
            if (lane == 0) atomicMin(thr + row0 + r, __float_as_uint(s_T[r]));
            r = rn;
#pragma unroll
            for (int u = 0; u < kAffPer; ++u) en[u] = nx[u];
        }
        __syncthreads();
        if (tid < kAffRows) s_T[tid] = fminf(s_T[tid], theirs);  // seen after the next barrier
    }
    // the lists as they stand (at most kAffHold entries each): the refinement merges and thins them
    if (tid < kAffRows && row0 + tid < n) {
        ccount[lists + row0 + tid] = s_cnt[tid] | (s_over[tid] ? kAffOver : 0u);
    }
}

// ---------------------------------------------------------------------------------------------
// exact selection (one wave per row): the row's lists over the column ranges merged to the
// columns whose lower bound is at most the k-th smallest upper bound of them all, then FP64
// distances of those from the FP32 inputs and the k smallest by (distance, index), ascending.
// Bound by the reads of the candidates' rows (n k dim 4 bytes from the caches); four candidates
// at a time keep their loads in flight and share the reduction across the lanes (20,000 points in
// 784-D, k = 90: 1.81 -> 1.13 ms).
// ---------------------------------------------------------------------------------------------
constexpr int kAffBatch = 4;
__global__ __launch_bounds__(kBlock) void k_aff_refine(const float* __restrict__ X, uint32_t n,
                                                       uint32_t dim, uint32_t dp, uint32_t k,
                                                       uint32_t splits, AffPoints P,
                                                       const uint2* __restrict__ cand,
                                                       const uint32_t* __restrict__ ccount,
                                                       uint32_t* __restrict__ idx,
                                                       double* __restrict__ d2,
                                                       uint32_t* __restrict__ overflow) {
    __shared__ double s_d[kWavesPerBlock][kAffKeep];
    __shared__ uint32_t s_j[kWavesPerBlock][kAffKeep];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t i = blockIdx.x * kWavesPerBlock + w;
    if (i >= n) return;
    uint32_t c = 0;
    {
        constexpr int kPer = kAffHold / kWave;  // entries per lane and list
        const float kd = aff_kdelta(dp), ni = P.nh[i], ai = P.ah[i], ei = P.eb[i];
        uint32_t j[kAffMaxSplits * kPer], hb[kAffMaxSplits * kPer];
        float lo[kAffMaxSplits * kPer];
        bool v[kAffMaxSplits * kPer];
        uint32_t over = 0;
#pragma unroll
        for (int s = 0; s < (int)kAffMaxSplits; ++s) {
            const uint32_t cf = s < (int)splits ? ccount[(size_t)s * n + i] : 0u;
            const uint32_t cs = cf & ~kAffOver;
            over |= cf & kAffOver;
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const size_t o = ((size_t)s * n + i) * kAffCap + lane + 64 * u;
                const int x = s * kPer + u;
                v[x] = (uint32_t)(lane + 64 * u) < cs;
                const uint2 en = v[x] ? cand[o] : make_uint2(i, 0u);
                float hi;
                aff_bounds(__uint_as_float(en.y), kd, ni, ai, ei, P.nh[en.x], P.ah[en.x],
                           P.eb[en.x], lo[x], hi);
                j[x] = en.x;
                hb[x] = __float_as_uint(hi);
            }
        }
        const float t = __uint_as_float(aff_kth<kAffMaxSplits * kPer>(hb, v, k, 32));
#pragma unroll
        for (int x = 0; x < (int)kAffMaxSplits * kPer; ++x) {
            const bool keep = v[x] && lo[x] <= t;
            const uint64_t bm = __ballot(keep);
            const uint32_t p = c + (uint32_t)__popcll(bm & lane_mask_lt());
            if (keep && p < kAffKeep) s_j[w][p] = j[x];
            c += (uint32_t)__popcll(bm);
        }
        if (lane == 0 && (over || c > kAffKeep || c < k)) atomicAdd(overflow, 1u);  // once a row
        c = min(c, kAffKeep);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* xi = X + (size_t)i * dim;
    for (uint32_t q = 0; q < c; q += kAffBatch) {
        const float* xj[kAffBatch];
        double s[kAffBatch];
#pragma unroll
        for (int u = 0; u < kAffBatch; ++u) {
            xj[u] = X + (size_t)s_j[w][min(q + u, c - 1)] * dim;
            s[u] = 0.0;
        }
#pragma unroll 4
        for (uint32_t e = lane; e < dim; e += kWave) {
            const double a = xi[e];
#pragma unroll
            for (int u = 0; u < kAffBatch; ++u) {
                const double df = a - (double)xj[u][e];
                s[u] = fma(df, df, s[u]);
            }
        }
        // sums over the lanes: halves and quarters of the wave take over one candidate each
        static_assert(kAffBatch == 4, "two exchange steps");
        const bool h = lane & 32, qd = lane & 16;
        const double a0 = h ? s[2] : s[0], a1 = h ? s[3] : s[1];
        const double b0 = h ? s[0] : s[2], b1 = h ? s[1] : s[3];
        const double p0 = a0 + __shfl_xor(b0, 32, kWave), p1 = a1 + __shfl_xor(b1, 32, kWave);
        double r = (qd ? p1 : p0) + __shfl_xor(qd ? p0 : p1, 16, kWave);
        for (int o = 8; o > 0; o >>= 1) r += __shfl_xor(r, o, kWave);
        const uint32_t at = q + (h ? 2u : 0u) + (qd ? 1u : 0u);
        if ((lane & 15) == 0 && at < c) s_d[w][at] = r;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (uint32_t q = lane; q < c; q += kWave) {
        const double dq = s_d[w][q];
        const uint32_t jq = s_j[w][q];
        uint32_t rank = 0;
        for (uint32_t p = 0; p < c; ++p) {
            const double dp_ = s_d[w][p];
            rank += (dp_ < dq || (dp_ == dq && s_j[w][p] < jq)) ? 1u : 0u;
        }
        if (rank < k) {
            idx[(size_t)i * k + rank] = jq;
            d2[(size_t)i * k + rank] = dq;
        }
    }
    // a row with fewer candidates than neighbours is reported; what follows still reads whole rows
    for (uint32_t q = c + lane; q < k; q += kWave) {
        idx[(size_t)i * k + q] = i;
        d2[(size_t)i * k + q] = 0.0;
    }
}

// ---------------------------------------------------------------------------------------------
// bandwidths: p_{j|i} = exp(-beta_i (d2_ij - d2_i0)) / sum, beta_i bisected until the entropy
// (natural log) is within tol of log(perplexity) (one wave per row, FP64; the scheme of
// openTSNE's binary search: doubling / halving until bracketed, then midpoints)
// ---------------------------------------------------------------------------------------------
constexpr int kAffMaxK = 128;
__global__ __launch_bounds__(kBlock) void k_aff_bandwidth(const double* __restrict__ d2,
                                                          uint32_t n, uint32_t k, double target,
                                                          double tol, int max_iter,
                                                          double* __restrict__ P,
                                                          double* __restrict__ beta_out) {
    const int lane = threadIdx.x & 63;
    const uint32_t i = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (i >= n) return;
    const double* row = d2 + (size_t)i * k;
    const double d0 = row[0];
    double dr[kAffMaxK / kWave];
    bool v[kAffMaxK / kWave];
#pragma unroll
    for (int u = 0; u < kAffMaxK / kWave; ++u) {
        const uint32_t q = lane + kWave * u;
        v[u] = q < k;
        dr[u] = v[u] ? row[q] - d0 : 0.0;
    }
    double beta = 1.0, lo = -__builtin_huge_val(), hi = __builtin_huge_val();
    double p[kAffMaxK / kWave];
    for (int it = 0; it < max_iter; ++it) {
        double e[kAffMaxK / kWave], s = 0.0;
#pragma unroll
        for (int u = 0; u < kAffMaxK / kWave; ++u) {
            e[u] = v[u] ? exp(-beta * dr[u]) : 0.0;
            s += e[u];
        }
        s = wave_sum_d(s);
        double h = 0.0;
#pragma unroll
        for (int u = 0; u < kAffMaxK / kWave; ++u) {
            p[u] = e[u] / s;
            h += dr[u] * p[u];
        }
        h = log(s) + beta * wave_sum_d(h);
        const double diff = h - target;
        if (fabs(diff) < tol) break;
        if (diff > 0.0) {  // entropy too high: sharpen
            lo = beta;
            beta = __builtin_isinf(hi) ? beta * 2.0 : 0.5 * (beta + hi);
        } else {
            hi = beta;
            beta = __builtin_isinf(lo) ? beta * 0.5 : 0.5 * (beta + lo);
        }
    }
#pragma unroll
    for (int u = 0; u < kAffMaxK / kWave; ++u)
        if (v[u]) P[(size_t)i * k + lane + kWave * u] = p[u];
    if (lane == 0) beta_out[i] = beta;
}

// ---------------------------------------------------------------------------------------------
// symmetrisation: entries (i, j, p_{j|i}) and (j, i, p_{j|i}) keyed by row * n + column, sorted
// by the project's sort (launch_sort: stable), equal keys (at most two) summed in FP64 in sorted
// order
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_sym_entries(const uint32_t* __restrict__ idx,
                                                        uint32_t n, uint32_t k,
                                                        uint64_t* __restrict__ keys,
                                                        uint32_t* __restrict__ vals) {
    const uint64_t nk = (uint64_t)n * k;
    const uint64_t e = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= nk) return;
    const uint64_t i = e / k, j = idx[e];
    keys[e] = i * n + j;
    keys[nk + e] = j * n + i;
    vals[e] = (uint32_t)e;
    vals[nk + e] = (uint32_t)(nk + e);
}

__global__ __launch_bounds__(kBlock) void k_sym_heads(const uint64_t* __restrict__ keys,
                                                      uint32_t m, uint32_t* __restrict__ head) {
    const uint32_t u = blockIdx.x * kBlock + threadIdx.x;
    if (u >= m) return;
    head[u] = (u == 0 || keys[u] != keys[u - 1]) ? 1u : 0u;
}

__global__ __launch_bounds__(kBlock) void k_sym_reduce(const uint64_t* __restrict__ keys,
                                                       const uint32_t* __restrict__ vals,
                                                       const uint32_t* __restrict__ pos,
                                                       uint32_t m, uint32_t n, uint32_t nk,
                                                       const double* __restrict__ P,
                                                       uint32_t* __restrict__ col,
                                                       float* __restrict__ val,
                                                       uint32_t* __restrict__ row_ptr,
                                                       const uint32_t* __restrict__ nnz) {
    const uint32_t u = blockIdx.x * kBlock + threadIdx.x;
    if (u >= m) return;
    const uint64_t key = keys[u];
    if (u > 0 && keys[u - 1] == key) return;  // not the first of its key
    const double two_n = 2.0 * (double)n;
    double s = P[vals[u] % nk] / two_n;
    if (u + 1 < m && keys[u + 1] == key) s += P[vals[u + 1] % nk] / two_n;
    const uint32_t q = pos[u];
    const uint64_t r64 = key / n;
    if (r64 >= n) return;  // no key of an entry: left behind by a sort that gave up (reported)
    const uint32_t r = (uint32_t)r64;
    col[q] = (uint32_t)(key % n);
    val[q] = (float)s;
    if (u == 0 || (uint32_t)(keys[u - 1] / n) != r) row_ptr[r] = q;  // every row has entries
    if (u == 0) row_ptr[n] = *nnz;
}

// ---------------------------------------------------------------------------------------------
uint32_t aff_dim_padded(uint32_t dim) { return div_up_a(dim, kAffKC) * kAffKC; }
uint32_t aff_cap() { return kAffCap; }
uint32_t aff_keep() { return kAffKeep; }

// Column ranges: one where the row blocks fill the 256 compute units about twice, else as many
// (up to kAffMaxSplits, at least two tiles each) as bring them there: 20,000 points are 157 row
// blocks, one per compute unit, so a single range would leave 99 units idle.
uint32_t aff_splits(uint32_t n) {
    const uint32_t rb = div_up_a(n, kAffRows), tiles = div_up_a(n, kAffCols);
    uint32_t s = 512u / rb;
    if (s > kAffMaxSplits) s = kAffMaxSplits;
    if (s > tiles / 2) s = tiles / 2;
    return s ? s : 1u;
}

void launch_aff_maxbits(hipStream_t s, const float* x, uint64_t n, uint32_t* out) {
    const uint32_t g = div_up_a(n, 8 * kBlock);
    k_aff_maxbits<<<g < 2048 ? g : 2048, kBlock, 0, s>>>((const uint32_t*)x, n, out);
}
void launch_aff_pack(hipStream_t s, const float* X, uint32_t n, uint32_t dim, float2 scale,
                     _Float16* Xh, float* nh, float* ah, float* eb) {
    k_aff_pack<<<div_up_a(n, kWavesPerBlock), kBlock, 0, s>>>(X, n, dim, aff_dim_padded(dim),
                                                              scale, Xh, nh, ah, eb);
}
void launch_aff_candidates(hipStream_t s, const _Float16* Xh, const float* nh, const float* ah,
                           const float* eb, uint32_t n, uint32_t dim, uint32_t k, uint32_t splits,
                           uint2* cand, uint32_t* ccount, uint32_t* thr) {
    const dim3 g(div_up_a(n, kAffRows), splits);
    k_aff_candidates<<<g, kAffThreads, 0, s>>>(Xh, nh, ah, eb, n, aff_dim_padded(dim), k, cand,
                                               ccount, thr);
}
void launch_aff_refine(hipStream_t s, const float* X, const float* nh, const float* ah,
                       const float* eb, uint32_t n, uint32_t dim, uint32_t k, uint32_t splits,
                       const uint2* cand, const uint32_t* ccount, uint32_t* idx, double* d2,
                       uint32_t* overflow) {
    k_aff_refine<<<div_up_a(n, kWavesPerBlock), kBlock, 0, s>>>(
        X, n, dim, aff_dim_padded(dim), k, splits, AffPoints{nh, ah, eb}, cand, ccount, idx, d2,
        overflow);
}
void launch_aff_bandwidth(hipStream_t s, const double* d2, uint32_t n, uint32_t k, double target,
                          double tol, int max_iter, double* P, double* beta) {
    k_aff_bandwidth<<<div_up_a(n, kWavesPerBlock), kBlock, 0, s>>>(d2, n, k, target, tol,
                                                                   max_iter, P, beta);
}
void launch_sym_entries(hipStream_t s, const uint32_t* idx, uint32_t n, uint32_t k,
                        uint64_t* keys, uint32_t* vals) {
    k_sym_entries<<<div_up_a((uint64_t)n * k, kBlock), kBlock, 0, s>>>(idx, n, k, keys, vals);
}
void launch_sym_heads(hipStream_t s, const uint64_t* keys, uint32_t m, uint32_t* head) {
    k_sym_heads<<<div_up_a(m, kBlock), kBlock, 0, s>>>(keys, m, head);
}
void launch_sym_reduce(hipStream_t s, const uint64_t* keys, const uint32_t* vals,
                       const uint32_t* pos, uint32_t m, uint32_t n, uint32_t nk, const double* P,
                       uint32_t* col, float* val, uint32_t* row_ptr, const uint32_t* nnz) {
    k_sym_reduce<<<div_up_a(m, kBlock), kBlock, 0, s>>>(keys, vals, pos, m, n, nk, P, col, val,
                                                        row_ptr, nnz);
}

}  // namespace bh
