// t-SNE gradient step on gfx950 (the TSNE driver of the reference, tsne.h:179-233, 272-301,
// 356-460), built on the Barnes-Hut repulsion of this library.
//
// The embedding lives in the caller's point order (P is indexed that way). Per iteration: the
// embedding as the solver's particles (staged by the first iteration of a call, then left by the
// update before), the tree, the walk with the t-SNE kernel (repulsion and per-point Z terms in sorted
// order) beside the CSR attraction on a stream of its own, the repulsion back in the caller's order
// with partial sums of Z in FP64, and one kernel that finishes Z and applies the momentum update
// y' = y + lr d + mu (y - y_prev).
#include "bh_common.h"
#include "bh_launch.h"

namespace bh {

__global__ __launch_bounds__(kBlock) void k_copy2(uint32_t n, const float* __restrict__ a,
                                                  const float* __restrict__ b,
                                                  float* __restrict__ ao, float* __restrict__ bo) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    ao[i] = a[i];
    bo[i] = b[i];
}

// embedding -> solver particles (unit masses, identity ids)
__global__ __launch_bounds__(kBlock) void k_tsne_stage(const float* __restrict__ yx,
                                                       const float* __restrict__ yy, uint32_t n,
                                                       float* __restrict__ x, float* __restrict__ y,
                                                       float* __restrict__ m,
                                                       uint32_t* __restrict__ id,
                                                       float2* __restrict__ xy) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float a = yx[i], b = yy[i];
    x[i] = a;
    y[i] = b;
    xy[i] = make_float2(a, b);
    m[i] = 1.0f;
    id[i] = i;
}

// One wave per row i: attraction exag * sum_j P_ij w_ij (y_j - y_i) with w = 1/(1+|y_j-y_i|^2)
// (updateAttractive, tsne.h:356-381). It needs only the current embedding, so it runs on a
// stream of its own beside the walk. The neighbours' positions are gathered
// from the interleaved copy xy (one 8-byte load per non-zero instead of two 4-byte ones: the
// gathers, not the bytes, bound this kernel).
__global__ __launch_bounds__(kBlock) void k_tsne_attract(const uint32_t* __restrict__ row_ptr,
                                                         const uint32_t* __restrict__ col,
                                                         const float* __restrict__ val, uint32_t n,
                                                         const float2* __restrict__ xy, float exag,
                                                         float* __restrict__ att_x,
                                                         float* __restrict__ att_y) {
    const int lane = threadIdx.x & 63;
    const uint32_t r = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (r >= n) return;
    const float2 yi = xy[r];
    float sx = 0.f, sy = 0.f;
    const uint32_t e0 = row_ptr[r], e1 = row_ptr[r + 1];
    for (uint32_t e = e0 + lane; e < e1; e += kWave) {
        const float2 yc = xy[col[e]];
        const float ddx = yc.x - yi.x, ddy = yc.y - yi.y;
        const float q = __builtin_amdgcn_rcpf(1.0f + fmaf(ddx, ddx, ddy * ddy));
        const float s = exag * val[e] * q;
        sx = fmaf(s, ddx, sx);
        sy = fmaf(s, ddy, sy);
    }
    sx = wave_sum_f(sx);
    sy = wave_sum_f(sy);
    if (lane != 0) return;
    att_x[r] = sx;
    att_y[r] = sy;
}

// derivative d_i = (s/Z) rep_i + attraction with s = 4 (updateRepulsive scaling,
// tsne.h:291-294; 1 in the reference's GPU step, nBodySolverGpuBH.cu:424), then
// y' = y + lr d + mu (y - y_prev) (updatePoints, tsne.h:179-206); one thread per point
// The update, and the next iteration's start where one follows (sx not null): its particles (the
// masses and indices stay those of the first stage), the interleaved copy and the partial bounds.
// Z comes as nz partial sums, which every block adds in the same order. Unsorting with Z's partial
// sums and this kernel stand for six launches of about 5 us each (partial sums, their sum, unsort,
// update, stage, bounds), a tenth of an iteration at 70k points.
__global__ __launch_bounds__(kBlock) void k_tsne_update(
    uint32_t n, const float* __restrict__ yx, const float* __restrict__ yy,
    const float* __restrict__ pyx, const float* __restrict__ pyy, const float* __restrict__ rep_x,
    const float* __restrict__ rep_y, const float* __restrict__ att_x,
    const float* __restrict__ att_y, const double* zpart, uint32_t nz, double* z_out,
    double rep_scale, float lr, float mu, float* __restrict__ nyx, float* __restrict__ nyy,
    float* __restrict__ dx_out, float* __restrict__ dy_out, float* __restrict__ sx,
    float* __restrict__ sy, float2* __restrict__ xy, float4* __restrict__ bounds) {
    double z = 0.0;
    for (uint32_t b = threadIdx.x; b < nz; b += kBlock) z += zpart[b];
    z = block_sum_d(z);
    if (blockIdx.x == 0 && threadIdx.x == 0 && z_out) *z_out = z;
    const float scale = (float)(rep_scale / z);
    float4 box = make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY);
    for (uint32_t r = blockIdx.x * kBlock + threadIdx.x; r < n; r += gridDim.x * kBlock) {
        const float dx = fmaf(scale, rep_x[r], att_x[r]);
        const float dy = fmaf(scale, rep_y[r], att_y[r]);
        if (dx_out) {
            dx_out[r] = dx;
            dy_out[r] = dy;
        }
        const float xi = yx[r], yi = yy[r];
        const float x = fmaf(lr, dx, xi) + mu * (xi - pyx[r]);
        const float y = fmaf(lr, dy, yi) + mu * (yi - pyy[r]);
        nyx[r] = x;
        nyy[r] = y;
        if (sx) {
            sx[r] = x;
            sy[r] = y;
            xy[r] = make_float2(x, y);
            box = minmax4(box, bounds_item(x, y));
        }
    }
    if (!sx) return;
    box = block_minmax4(box);
    if (threadIdx.x == 0) bounds[blockIdx.x] = box;
}

// ------------------------------------------------------------------------------------------
// Exact Z of an embedding (unit masses): sum over ordered pairs of 1 / (1 + |y_i - y_j|^2), FP64.
// Every unordered pair of tiles of kZTile points is one item of work, counted twice (a diagonal
// tile once); within it a thread holds two rows and runs over the columns in LDS. The two terms
// of a column share one reciprocal, 1/a + 1/b = (a + b) / (a b): a and b are at least 1 and at
// most 1e78 for FP32 positions, so the product neither under- nor overflows. The reciprocal
// estimate (relative error 4.6e-8) takes two Newton steps, which leave rounding only. Diagonal
// tiles and the ragged last one take each term by itself, masked.
// FP64 VALU bound: 15 full-rate FP64 operations and one estimate per two pairs, each pair once.
// 70,000 points: the whole cost call 5.48 -> 1.00 ms.
// Before: every ordered pair with an IEEE division, through per-sink sums of forces too.
// ------------------------------------------------------------------------------------------
constexpr int kZTile = 256;
constexpr int kZThreads = kZTile / 2;
constexpr uint32_t kZMaxBlocks = 4096;

__device__ __forceinline__ double rcp_newton2(double v) {
    double r = __builtin_amdgcn_rcp(v);
    r = fma(r, fma(-v, r, 1.0), r);
    return fma(r, fma(-v, r, 1.0), r);
}

__global__ __launch_bounds__(kZThreads) void k_tsne_z(const float4* __restrict__ pos4, uint32_t n,
                                                      double* __restrict__ partials) {
    __shared__ double2 s_q[kZTile];
    __shared__ double red[kZThreads / kWave];
    const int tid = threadIdx.x;
    const uint64_t nt = (n + kZTile - 1) / kZTile, items = nt * (nt + 1) / 2;
    double acc = 0.0;
    for (uint64_t it = blockIdx.x; it < items; it += gridDim.x) {
        // item -> (I, J), I <= J: column J starts at item J (J + 1) / 2
        uint64_t J = (uint64_t)((sqrt(8.0 * (double)it + 1.0) - 1.0) * 0.5);
        while (J * (J + 1) / 2 > it) --J;
        while ((J + 1) * (J + 2) / 2 <= it) ++J;
        const uint64_t I = it - J * (J + 1) / 2;
        const uint32_t i0 = (uint32_t)I * kZTile + tid, i1 = i0 + kZThreads;
        const uint32_t j0 = (uint32_t)J * kZTile;
        __syncthreads();  // the previous item's columns are read
        for (int c = tid; c < kZTile; c += kZThreads) {
            const float4 q = pos4[min(j0 + c, n - 1)];
            s_q[c] = make_double2(q.x, q.y);
        }
        const float4 f0 = pos4[min(i0, n - 1)], f1 = pos4[min(i1, n - 1)];
        const double x0 = f0.x, y0 = f0.y, x1 = f1.x, y1 = f1.y;
        __syncthreads();
        double s = 0.0;
        if (I != J && j0 + kZTile <= n) {  // block-uniform
#pragma unroll 4
            for (int c = 0; c < kZTile; ++c) {
                const double2 q = s_q[c];
                const double dx0 = q.x - x0, dy0 = q.y - y0, dx1 = q.x - x1, dy1 = q.y - y1;
                const double a = fma(dx0, dx0, fma(dy0, dy0, 1.0));
                const double b = fma(dx1, dx1, fma(dy1, dy1, 1.0));
                s = fma(a + b, rcp_newton2(a * b), s);
            }
            s *= 2.0;
        } else {
            const uint32_t cols = min((uint32_t)kZTile, n - j0);
            for (uint32_t c = 0; c < cols; ++c) {
                const double2 q = s_q[c];
                const double dx0 = q.x - x0, dy0 = q.y - y0, dx1 = q.x - x1, dy1 = q.y - y1;
                const double a = fma(dx0, dx0, fma(dy0, dy0, 1.0));
                const double b = fma(dx1, dx1, fma(dy1, dy1, 1.0));
                if (i0 < n && j0 + c != i0) s += rcp_newton2(a);
                if (i1 < n && j0 + c != i1) s += rcp_newton2(b);
            }
            if (I != J) s *= 2.0;
        }
        acc += s;
    }
    acc = wave_sum_d(acc);
    if ((tid & 63) == 0) red[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) {
        double b = 0.0;
        for (int k = 0; k < kZThreads / kWave; ++k) b += red[k];
        partials[blockIdx.x] = b;
    }
}

// KL divergence sum_{i != j} P_ij log2(P_ij / Q_ij), Q_ij = w_ij / Z, in FP64
// (costFunction, tsne.h:383-460); block partials, summed in order by k_tsne_kl_final.
__global__ __launch_bounds__(kBlock) void k_tsne_kl(const uint32_t* __restrict__ row_ptr,
                                                    const uint32_t* __restrict__ col,
                                                    const float* __restrict__ val, uint32_t n,
                                                    const float* __restrict__ yx,
                                                    const float* __restrict__ yy,
                                                    const double* __restrict__ z,
                                                    double* __restrict__ partials) {
    __shared__ double red[kWavesPerBlock];
    const double Z = *z;
    double acc = 0.0;
    for (uint32_t r = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6); r < n;
         r += gridDim.x * kWavesPerBlock) {
        const double xi = yx[r], yi = yy[r];
        for (uint32_t e = row_ptr[r] + (threadIdx.x & 63); e < row_ptr[r + 1]; e += kWave) {
            const uint32_t c = col[e];
            if (c == r) continue;
            const double ddx = (double)yx[c] - xi, ddy = (double)yy[c] - yi;
            const double p = val[e];  // P / Q = P Z (1 + |y_i - y_j|^2)
            acc += p * log2(p * Z * (1.0 + (ddx * ddx + ddy * ddy)));
        }
    }
    acc = wave_sum_d(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = 0.0;
        for (int k = 0; k < kWavesPerBlock; ++k) b += red[k];
        partials[blockIdx.x] = b;
    }
}

__global__ __launch_bounds__(kBlock) void k_sum_f64(const double* __restrict__ v, uint32_t nv,
                                                    double* __restrict__ out) {
    __shared__ double red[kWavesPerBlock];
    double s = 0.0;
    for (uint32_t b = threadIdx.x; b < nv; b += kBlock) s += v[b];
    s = wave_sum_d(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = 0.0;
        for (int k = 0; k < kWavesPerBlock; ++k) b += red[k];
        *out = b;
    }
}

static inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

void launch_tsne_stage(hipStream_t s, const float* yx, const float* yy, uint32_t n, float* x,
                       float* y, float* m, uint32_t* id, float2* xy) {
    k_tsne_stage<<<div_up(n, kBlock), kBlock, 0, s>>>(yx, yy, n, x, y, m, id, xy);
}

void launch_copy2(hipStream_t s, uint32_t n, const float* a, const float* b, float* ao, float* bo) {
    if (n) k_copy2<<<div_up(n, kBlock), kBlock, 0, s>>>(n, a, b, ao, bo);
}

void launch_tsne_attract(hipStream_t s, const uint32_t* row_ptr, const uint32_t* col,
                         const float* val, uint32_t n, const float2* xy, float exag, float* att_x,
                         float* att_y) {
    k_tsne_attract<<<div_up(n, kWavesPerBlock), kBlock, 0, s>>>(row_ptr, col, val, n, xy, exag,
                                                                att_x, att_y);
}

void launch_tsne_update(hipStream_t s, uint32_t n, const float* yx, const float* yy,
                        const float* pyx, const float* pyy, const float* rep_x, const float* rep_y,
                        const float* att_x, const float* att_y, const double* zpart, uint32_t nz,
                        double* z_out, double rep_scale, float lr, float mu, float* nyx, float* nyy,
                        float* dx, float* dy, float* sx, float* sy, float2* xy, float4* bounds) {
    k_tsne_update<<<update_blocks(n), kBlock, 0, s>>>(
        n, yx, yy, pyx, pyy, rep_x, rep_y, att_x, att_y, zpart, nz, z_out, rep_scale, lr, mu, nyx,
        nyy, dx, dy, sx, sy, xy, bounds);
}

uint32_t tsne_kl_blocks(uint32_t n) {
    uint32_t g = div_up(n, kWavesPerBlock);
    return g > kMaxReduceBlocks ? kMaxReduceBlocks : (g ? g : 1);
}

void launch_tsne_kl(hipStream_t s, const uint32_t* row_ptr, const uint32_t* col, const float* val,
                    uint32_t n, const float* yx, const float* yy, const double* z,
                    double* partials, double* out) {
    const uint32_t g = tsne_kl_blocks(n);
    k_tsne_kl<<<g, kBlock, 0, s>>>(row_ptr, col, val, n, yx, yy, z, partials);
    k_sum_f64<<<1, kBlock, 0, s>>>(partials, g, out);
}

uint32_t tsne_z_blocks(uint32_t n) {
    const uint64_t nt = div_up(n, kZTile), items = nt * (nt + 1) / 2;
    return items < kZMaxBlocks ? (uint32_t)items : kZMaxBlocks;
}

void launch_tsne_z(hipStream_t s, const float4* pos4, uint32_t n, double* partials, double* z) {
    const uint32_t g = tsne_z_blocks(n);
    k_tsne_z<<<g, kZThreads, 0, s>>>(pos4, n, partials);
    k_sum_f64<<<1, kBlock, 0, s>>>(partials, g, z);
}

}  // namespace bh
