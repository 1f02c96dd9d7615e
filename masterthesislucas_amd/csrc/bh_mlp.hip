// Learned far-field correction on gfx950: training data from the tree itself, hand-written
// forward / backward / Adam kernels (FP32), and BF16 MFMA inference (FP32 accumulation).
//
// Data set: for sampled sinks, the cells the opening-angle test accepts (within a band of
// l / r) are collected by a per-sink stackless walk over the pre-order tree, then each
// (sink, cell) pair is labelled by an FP64 sum over the cell's particles minus the FP64
// monopole, in units of M l^2 / r^4 (bh_mlp.h). Training minimises the mean squared error over
// all outputs with Adam; gradients are reduced per chunk of samples and then summed in a fixed
// order, so a training run is deterministic.
#include "bh_common.h"
#include "bh_launch.h"
#include "bh_mlp.h"

namespace bh {

static inline uint32_t div_up_u(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// ---------------------------------------------------------------------------------------------
// parameters -> MFMA operand layout
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_mlp_prep_bf16(const float* __restrict__ p,
                                                      MlpBf16* __restrict__ W) {
    const int lane = threadIdx.x;
    const int r16 = lane & 15, q4 = lane >> 4;
    const float* W1 = p + kMlpOffW1;
    const float* b1 = p + kMlpOffB1;
    const float* W2 = p + kMlpOffW2;
    const float* W3 = p + kMlpOffW3;
    for (int u = 0; u < 4; ++u) {
        bf16x4 v;
        for (int i = 0; i < 4; ++i) {
            const int in = 4 * q4 + i, unit = 16 * u + r16;
            float w = 0.f;
            if (in < kMlpIn) w = W1[in * kMlpH + unit];
            else if (in == kMlpIn) w = b1[unit];  // constant-1 input carries the bias
            v[i] = f32_to_bf16(w);
        }
        W->w1[u][lane] = v;
    }
    for (int u = 0; u < 4; ++u)
        for (int c = 0; c < 2; ++c) {
            bf16x8 v;
            for (int j = 0; j < 8; ++j)
                v[j] = (__bf16)W2[mlp_unit_of(c, 8 * q4 + j) * kMlpH + 16 * u + r16];
            W->w2[u][c][lane] = v;
        }
    for (int c = 0; c < 2; ++c) {
        bf16x8 v;
        for (int j = 0; j < 8; ++j)
            v[j] = (__bf16)(r16 < kMlpOut ? W3[mlp_unit_of(c, 8 * q4 + j) * kMlpOut + r16] : 0.f);
        W->w3[c][lane] = v;
    }
    W->b2[lane] = p[kMlpOffB2 + lane];
    if (lane < 16) W->b3[lane] = lane < kMlpOut ? p[kMlpOffB3 + lane] : 0.f;
}

// stage the BF16 weights in LDS once per block
__device__ __forceinline__ void stage_weights(const MlpBf16* __restrict__ W, MlpBf16* ws) {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(W);
    uint32_t* dst = reinterpret_cast<uint32_t*>(ws);
    for (uint32_t i = threadIdx.x; i < sizeof(MlpBf16) / 4; i += kBlock) dst[i] = src[i];
}

// one wave: features of 64 rows (stride `stride` floats, the first kMlpIn used) -> the 14
// outputs of each row in LDS (ys[64][16])
__device__ __forceinline__ void infer_rows(const MlpBf16* ws, const float* __restrict__ X,
                                           uint32_t base, uint32_t n, uint32_t stride, short* xs,
                                           float* ys) {
    const int lane = threadIdx.x & 63;
    const uint32_t i = base + lane;
    short* row = xs + lane * kMlpInPad;
#pragma unroll
    for (int c = 0; c < kMlpInPad; ++c) {
        float v = 0.f;
        if (c < kMlpIn) v = i < n ? X[(size_t)i * stride + c] : 0.f;
        else if (c == kMlpIn) v = 1.f;
        row[c] = f32_to_bf16(v);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    f32x4 out[4];
    mlp_wave_infer(ws, xs, out);
    const int r16 = lane & 15, q4 = lane >> 4;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) ys[(16 * s + r16) * 16 + 4 * q4 + e] = out[s][e];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------------------------
// inference: BF16 MFMA (one wave per 64 samples) and the FP32 reference forward
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_mlp_infer_bf16(const float* __restrict__ X, uint32_t n,
                                                           const MlpBf16* __restrict__ W,
                                                           float* __restrict__ Y) {
    __shared__ short xs[kWavesPerBlock][64 * kMlpInPad];
    __shared__ float ys[kWavesPerBlock][64 * 16];
    __shared__ MlpBf16 ws;
    stage_weights(W, &ws);
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t base = (blockIdx.x * kWavesPerBlock + w) * 64u;
    infer_rows(&ws, X, base, n, kMlpIn, xs[w], ys[w]);
    const uint32_t i = base + lane;
    if (i < n)
        for (int o = 0; o < kMlpOut; ++o) Y[(size_t)i * kMlpOut + o] = ys[w][lane * 16 + o];
}

// per node: the network on its features -> the walk's coefficient record
__global__ __launch_bounds__(kBlock) void k_cell_coefs(const float* __restrict__ feat,
                                                       const Node* __restrict__ nodes,
                                                       const BuildParams* __restrict__ prm,
                                                       uint32_t cap_nodes,
                                                       const MlpBf16* __restrict__ W,
                                                       float4* __restrict__ coef) {
    __shared__ short xs[kWavesPerBlock][64 * kMlpInPad];
    __shared__ float ys[kWavesPerBlock][64 * 16];
    __shared__ MlpBf16 ws;
    const uint32_t nn = min(prm->n_nodes, cap_nodes);
    if (blockIdx.x * (64u * kWavesPerBlock) >= nn) return;  // whole block: past the last node
    stage_weights(W, &ws);
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t base = (blockIdx.x * kWavesPerBlock + w) * 64u;
    if (base >= nn) return;  // wave-uniform
    infer_rows(&ws, feat, base, nn, kMlpIn, xs[w], ys[w]);
    const uint32_t k = base + lane;
    if (k >= nn) return;
    // the cell side as the walk takes it (the FP32 root side scaled by 2^-level, exact) and
    // M l^2 with the walk's rounding
    const Node nd = nodes[k];
    const float l = ldexpf(prm->side, -(int)(nd.meta & kMetaLevelMask));
    float r[kCoefStride];
    learned_record(&ys[w][lane * 16], nd.mass * l * l, l, r);
    float4* dst = coef + (size_t)k * (kCoefStride / 4);
#pragma unroll
    for (int q = 0; q < kCoefStride / 4; ++q)
        dst[q] = make_float4(r[4 * q], r[4 * q + 1], r[4 * q + 2], r[4 * q + 3]);
}

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + __expf(-v)); }
__device__ __forceinline__ float dsilu_f(float v) {
    const float s = 1.0f / (1.0f + __expf(-v));
    return s * (1.0f + v * (1.0f - s));
}

__global__ __launch_bounds__(kBlock) void k_mlp_forward_f32(const float* __restrict__ X, uint32_t n,
                                                            const float* __restrict__ p,
                                                            float* __restrict__ Y) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    float x[kMlpIn], a1[kMlpH], y[kMlpOut];
#pragma unroll
    for (int c = 0; c < kMlpIn; ++c) x[c] = X[(size_t)i * kMlpIn + c];
#pragma unroll
    for (int j = 0; j < kMlpH; ++j) {
        float z = p[kMlpOffB1 + j];
#pragma unroll
        for (int c = 0; c < kMlpIn; ++c) z = fmaf(x[c], p[kMlpOffW1 + c * kMlpH + j], z);
        a1[j] = silu_f(z);
    }
#pragma unroll
    for (int o = 0; o < kMlpOut; ++o) y[o] = p[kMlpOffB3 + o];
    for (int j = 0; j < kMlpH; ++j) {
        float z = p[kMlpOffB2 + j];
#pragma unroll
        for (int k = 0; k < kMlpH; ++k) z = fmaf(a1[k], p[kMlpOffW2 + k * kMlpH + j], z);
        const float a2 = silu_f(z);
#pragma unroll
        for (int o = 0; o < kMlpOut; ++o) y[o] = fmaf(a2, p[kMlpOffW3 + j * kMlpOut + o], y[o]);
    }
#pragma unroll
    for (int o = 0; o < kMlpOut; ++o) Y[(size_t)i * kMlpOut + o] = y[o];
}

// basis of the pair offset (complex, interleaved re/im): w, conj w, w^3, q, q w^2, q conj(w)^2,
// q w^4
__device__ __forceinline__ void learned_basis_f(float ux, float uy, float q, float* b) {
    const float w2r = fmaf(ux, ux, -uy * uy), w2i = 2.0f * ux * uy;
    const float w3r = fmaf(w2r, ux, -w2i * uy), w3i = fmaf(w2r, uy, w2i * ux);
    const float w4r = fmaf(w2r, w2r, -w2i * w2i), w4i = 2.0f * w2r * w2i;
    b[0] = ux; b[1] = uy;
    b[2] = ux; b[3] = -uy;
    b[4] = w3r; b[5] = w3i;
    b[6] = q; b[7] = 0.f;
    b[8] = q * w2r; b[9] = q * w2i;
    b[10] = q * w2r; b[11] = -q * w2i;
    b[12] = q * w4r; b[13] = q * w4i;
}

// ---------------------------------------------------------------------------------------------
// training: forward, backward and weight gradients of a batch in one kernel.
// A sample is a row of kLearnSample floats (10 cell features, w_x, w_y, q) and a label
// T[2]; its prediction is p = sum_j c_j b_j (complex) with c = the network's 14 outputs and b
// the basis of (w, q); loss = sum |p - T|^2 / (2 B).
//
// A block of four waves takes tiles of kTrainTile samples. Every product (three forward, two
// backward, three weight gradients) runs on the FP32 matrix instruction
// v_mfma_f32_16x16x4_f32, wave w owning the hidden units [16 w, 16 w + 16): its columns of W1,
// W2, W2^T and W3^T stay in registers, activations pass between the waves through LDS, and the
// weight gradients accumulate in registers over the block's tiles and are written once, as the
// block's partial (k_mlp_adam adds the partials in block order: deterministic).
//   D = A B of 16x16x4: A[row l % 16][k l / 16], B[k l / 16][col l % 16],
//   D[row 4 (l / 16) + e][col l % 16] in element e of lane l.
// Bound by latency (a 4,096-sample batch is 133 MFLOP, 0.9 us of matrix work on the whole chip):
// 128 blocks of 32 samples, no scratch in memory. Before: one thread per sample on 16 blocks
// (79 us) with the activations in memory, and a thread per parameter reading 1,024 samples one
// after the other (189 us).
// ---------------------------------------------------------------------------------------------
constexpr int kTrainTile = 32;            // samples per tile
constexpr uint32_t kTrainBlocks = 256;    // blocks (and gradient partials) of a large launch
constexpr uint32_t kTrainChain = 32;      // most tiles that a block's sums run over
constexpr int kActStride = kMlpH + 4;     // LDS row stride of activations (bank spread)
constexpr int kTrainX = 12;               // inputs padded to a multiple of 4; slot 10 holds 1

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <bool GRAD>
__global__ __launch_bounds__(kBlock) void k_mlp_train(const float* __restrict__ X,
                                                      const float* __restrict__ T,
                                                      const uint32_t* __restrict__ order,
                                                      uint32_t B, const float* __restrict__ p,
                                                      double* __restrict__ loss_part,
                                                      float* __restrict__ partials, int terms) {
    constexpr int ST = kTrainTile / 16;  // sample blocks of a tile
    __shared__ float s_x[kTrainTile][16 + 1];
    __shared__ float s_off[kTrainTile][5];  // w_x, w_y, q, label
    __shared__ float s_a1[kTrainTile][kActStride], s_a2[kTrainTile][kActStride];
    __shared__ float s_dz[kTrainTile][kActStride];
    __shared__ float s_y[kTrainTile][17];   // outputs, then their gradients
    __shared__ double s_sq[kTrainTile];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q4 = lane >> 4;
    const int unit = 16 * w + r;
    // this wave's weights as B operands
    float w1[kTrainX / 4], w2[kMlpH / 4], w2t[kMlpH / 4], w3t[4];
#pragma unroll
    for (int k = 0; k < kTrainX / 4; ++k) {
        const int in = 4 * k + q4;
        w1[k] = in < kMlpIn ? p[kMlpOffW1 + in * kMlpH + unit]
                            : (in == kMlpIn ? p[kMlpOffB1 + unit] : 0.f);
    }
#pragma unroll
    for (int k = 0; k < kMlpH / 4; ++k) {
        w2[k] = p[kMlpOffW2 + (4 * k + q4) * kMlpH + unit];
        if (GRAD) w2t[k] = p[kMlpOffW2 + unit * kMlpH + 4 * k + q4];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int o = 4 * k + q4;
        w3t[k] = GRAD && o < kMlpOut ? p[kMlpOffW3 + unit * kMlpOut + o] : 0.f;
    }
    float w3[kMlpH / 4];  // layer 3: output r, all units (waves 0 .. ST - 1 use it)
#pragma unroll
    for (int k = 0; k < kMlpH / 4; ++k)
        w3[k] = w < ST && r < kMlpOut ? p[kMlpOffW3 + (4 * k + q4) * kMlpOut + r] : 0.f;
    const float b2 = p[kMlpOffB2 + unit];
    const float b3 = r < kMlpOut ? p[kMlpOffB3 + r] : 0.f;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 g1 = zero, g3 = zero, g2[4] = {zero, zero, zero, zero};
    float gb2 = 0.f, gb3 = 0.f;
    double sq = 0.0;  // threads < kTrainTile: squared errors of their samples
    const float inv_b = 1.0f / (float)B;
    const uint32_t ntiles = (B + kTrainTile - 1) / kTrainTile;
    for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // stage the tile: 8 threads per sample, features (bias input 1 in slot 10) and offsets
        {
            const int smp = tid >> 3, part = tid & 7;
            const uint32_t i = tile * kTrainTile + smp;
            const bool live = i < B;
            const uint32_t src = live ? (order ? order[i] : i) : 0u;
            const float* row = X + (size_t)src * kLearnSample;
#pragma unroll
            for (int c = part; c < 16; c += 8)
                s_x[smp][c] = c < kMlpIn ? (live ? row[c] : 0.f) : (c == kMlpIn && live ? 1.f : 0.f);
            if (part < 5)
                s_off[smp][part] = !live ? 0.f
                                 : part < 3 ? row[kMlpIn + part] : T[(size_t)src * 2 + part - 3];
        }
        __syncthreads();
        // layer 1
        float d1[ST][4], d2[ST][4];
#pragma unroll
        for (int st = 0; st < ST; ++st) {
            f32x4 z = zero;
#pragma unroll
            for (int k = 0; k < kTrainX / 4; ++k) z = mfma4(s_x[16 * st + r][4 * k + q4], w1[k], z);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s_a1[16 * st + 4 * q4 + e][unit] = silu_f(z[e]);
                d1[st][e] = GRAD ? dsilu_f(z[e]) : 0.f;
            }
        }
        __syncthreads();
        // layer 2
        f32x4 z2[ST];
#pragma unroll
        for (int st = 0; st < ST; ++st) z2[st] = f32x4{b2, b2, b2, b2};
#pragma unroll
        for (int k = 0; k < kMlpH / 4; ++k)
#pragma unroll
            for (int st = 0; st < ST; ++st)
                z2[st] = mfma4(s_a1[16 * st + r][4 * k + q4], w2[k], z2[st]);
#pragma unroll
        for (int st = 0; st < ST; ++st)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s_a2[16 * st + 4 * q4 + e][unit] = silu_f(z2[st][e]);
                d2[st][e] = GRAD ? dsilu_f(z2[st][e]) : 0.f;
            }
        __syncthreads();
        // layer 3: one sample block per wave
        if (w < ST) {
            f32x4 y0 = {b3, b3, b3, b3}, y1 = zero;
#pragma unroll
            for (int k = 0; k < kMlpH / 4; k += 2) {
                y0 = mfma4(s_a2[16 * w + r][4 * k + q4], w3[k], y0);
                y1 = mfma4(s_a2[16 * w + r][4 * k + 4 + q4], w3[k + 1], y1);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) s_y[16 * w + 4 * q4 + e][r] = y0[e] + y1[e];
        }
        __syncthreads();
        // prediction, error and output gradients of one sample per thread
        if (tid < kTrainTile) {
            float bas[kMlpOut];
            learned_basis_f(s_off[tid][0], s_off[tid][1], s_off[tid][2], bas);
            // a network trained with fewer terms: the basis beyond them is zero (no prediction,
            // no gradient)
#pragma unroll
            for (int o = 0; o < kMlpOut; ++o)
                if (o >= 2 * terms) bas[o] = 0.f;
            float pr = 0.f, pi = 0.f;
#pragma unroll
            for (int j = 0; j < kLearnTerms; ++j) {
                const float yr = s_y[tid][2 * j], yi = s_y[tid][2 * j + 1];
                pr = fmaf(yr, bas[2 * j], fmaf(-yi, bas[2 * j + 1], pr));
                pi = fmaf(yr, bas[2 * j + 1], fmaf(yi, bas[2 * j], pi));
            }
            const bool live = tile * kTrainTile + tid < B;
            const float ex = live ? pr - s_off[tid][3] : 0.f;
            const float ey = live ? pi - s_off[tid][4] : 0.f;
            sq += (double)ex * ex + (double)ey * ey;
            if (GRAD) {
                // dL/dRe c_j = Re(conj(e) b_j) / B, dL/dIm c_j = Im(conj(b_j) e) / B
#pragma unroll
                for (int j = 0; j < kLearnTerms; ++j) {
                    const float br = bas[2 * j], bi = bas[2 * j + 1];
                    s_y[tid][2 * j] = fmaf(ex, br, ey * bi) * inv_b;
                    s_y[tid][2 * j + 1] = fmaf(ey, br, -ex * bi) * inv_b;
                }
                s_y[tid][14] = s_y[tid][15] = 0.f;
            }
        }
        __syncthreads();
        if constexpr (GRAD) {
            // dz2 = (dy W3^T) * silu'(z2)
#pragma unroll
            for (int st = 0; st < ST; ++st) {
                f32x4 da = zero;
#pragma unroll
                for (int k = 0; k < 4; ++k) da = mfma4(s_y[16 * st + r][4 * k + q4], w3t[k], da);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s_dz[16 * st + 4 * q4 + e][unit] = da[e] * d2[st][e];
            }
            __syncthreads();
            // dz1 = (dz2 W2^T) * silu'(z1), kept until the reads of dz2 below are done
            f32x4 da[ST];
#pragma unroll
            for (int st = 0; st < ST; ++st) da[st] = zero;
#pragma unroll
            for (int k = 0; k < kMlpH / 4; ++k)
#pragma unroll
                for (int st = 0; st < ST; ++st)
                    da[st] = mfma4(s_dz[16 * st + r][4 * k + q4], w2t[k], da[st]);
            // dW2 (rows a1 units, columns this wave's units), dW3 (rows this wave's units), biases
#pragma unroll
            for (int k = 0; k < kTrainTile / 4; ++k) {
                const float bz = s_dz[4 * k + q4][unit];
#pragma unroll
                for (int t = 0; t < 4; ++t) g2[t] = mfma4(s_a1[4 * k + q4][16 * t + r], bz, g2[t]);
                g3 = mfma4(s_a2[4 * k + q4][unit], s_y[4 * k + q4][r], g3);
            }
            if (tid < kMlpH) {
#pragma unroll
                for (int s = 0; s < kTrainTile; ++s) gb2 += s_dz[s][tid];
            } else if (tid < kMlpH + kMlpOut) {
#pragma unroll
                for (int s = 0; s < kTrainTile; ++s) gb3 += s_y[s][tid - kMlpH];
            }
            __syncthreads();
#pragma unroll
            for (int st = 0; st < ST; ++st)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s_dz[16 * st + 4 * q4 + e][unit] = da[st][e] * d1[st][e];
            // dW1 and, in row 10, db1: this wave reads only the columns it wrote
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int k = 0; k < kTrainTile / 4; ++k)
                g1 = mfma4(s_x[4 * k + q4][r], s_dz[4 * k + q4][unit], g1);
        }
        __syncthreads();  // the next tile overwrites the staged samples
    }
    if (tid < kTrainTile) s_sq[tid] = sq;
    __syncthreads();
    if (tid == 0 && loss_part) {
        double s = 0.0;
        for (int k = 0; k < kTrainTile; ++k) s += s_sq[k];
        loss_part[blockIdx.x] = s;
    }
    if constexpr (GRAD) {
        float* out = partials + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 4 * q4 + e;
            if (row < kMlpIn) out[kMlpOffW1 + row * kMlpH + unit] = g1[e];
            if (row == kMlpIn) out[kMlpOffB1 + unit] = g1[e];
            if (r < kMlpOut) out[kMlpOffW3 + (16 * w + row) * kMlpOut + r] = g3[e];
#pragma unroll
            for (int t = 0; t < 4; ++t) out[kMlpOffW2 + (16 * t + row) * kMlpH + unit] = g2[t][e];
        }
        if (tid < kMlpH) out[kMlpOffB2 + tid] = gb2;
        else if (tid < kMlpH + kMlpOut) out[kMlpOffB3 + tid - kMlpH] = gb3;
    }
}

// Sum the block partials in order (kAdamGroups threads per parameter take every kAdamGroups-th
// partial, several loads in flight, and their sums are added in order); optionally export the
// gradient; Adam update. Latency bound: 128 partials of 5,774 parameters (3 MB).
constexpr int kAdamGroups = 16;
__global__ __launch_bounds__(64 * kAdamGroups) void k_mlp_adam(float* __restrict__ p,
                                                     const float* __restrict__ partials,
                                                     uint32_t nchunks, float* __restrict__ m1,
                                                     float* __restrict__ m2, float lr, float beta1,
                                                     float beta2, float eps, int step,
                                                     float* __restrict__ grad_out, int apply) {
    __shared__ float s_g[kAdamGroups][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int q = blockIdx.x * 64 + lane;
    float s = 0.f;
    if (q < kMlpParams) {
        constexpr uint32_t kUnroll = 8;
        for (uint32_t c0 = grp; c0 < nchunks; c0 += kUnroll * kAdamGroups) {
            float v[kUnroll];
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; ++u) {
                const uint32_t c = c0 + u * kAdamGroups;
                v[u] = c < nchunks ? partials[(size_t)c * kMlpParams + q] : 0.f;
            }
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; ++u) s += v[u];
        }
    }
    s_g[grp][lane] = s;
    __syncthreads();
    if (grp != 0 || q >= kMlpParams) return;
    float g = 0.f;
#pragma unroll
    for (int k = 0; k < kAdamGroups; ++k) g += s_g[k][lane];
    if (grad_out) grad_out[q] = g;
    if (!apply) return;
    const float a = m1[q] = beta1 * m1[q] + (1.f - beta1) * g;
    const float b = m2[q] = beta2 * m2[q] + (1.f - beta2) * g * g;
    const float bc1 = 1.f - __powf(beta1, (float)step), bc2 = 1.f - __powf(beta2, (float)step);
    p[q] -= lr * (a / bc1) / (sqrtf(b / bc2) + eps);
}

// Adam with a given gradient (host-provided), same update as above
__global__ __launch_bounds__(kBlock) void k_mlp_adam_grad(float* __restrict__ p,
                                                          const float* __restrict__ g_in,
                                                          float* __restrict__ m1,
                                                          float* __restrict__ m2, float lr,
                                                          float beta1, float beta2, float eps,
                                                          int step) {
    const int q = blockIdx.x * kBlock + threadIdx.x;
    if (q >= kMlpParams) return;
    const float g = g_in[q];
    const float a = m1[q] = beta1 * m1[q] + (1.f - beta1) * g;
    const float b = m2[q] = beta2 * m2[q] + (1.f - beta2) * g * g;
    const float bc1 = 1.f - __powf(beta1, (float)step), bc2 = 1.f - __powf(beta2, (float)step);
    p[q] -= lr * (a / bc1) / (sqrtf(b / bc2) + eps);
}

// ---------------------------------------------------------------------------------------------
// data set from the tree
// ---------------------------------------------------------------------------------------------
// Per sample sink (sorted index), a stackless pre-order walk with the traversal's own FP32
// acceptance test; accepted cells with d^2 <= l^2 / band^2 (l / r >= band) are recorded.
__global__ __launch_bounds__(kBlock) void k_collect_pairs(const float4* __restrict__ pos4,
                                                          const Node* __restrict__ nodes,
                                                          const BuildParams* __restrict__ prm,
                                                          const uint32_t* __restrict__ sinks,
                                                          uint32_t ns, float inv_theta2,
                                                          float inv_band2, uint32_t cap,
                                                          uint32_t* __restrict__ pairs,
                                                          uint32_t* __restrict__ counts) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= ns) return;
    const uint32_t nn = prm->n_nodes;
    const float4 me = pos4[sinks[t]];
    uint32_t k = 0, c = 0;
    while (k < nn) {
        const Node nd = nodes[k];
        const float dx = nd.cx - me.x, dy = nd.cy - me.y;
        const float d2 = fmaf(dx, dx, dy * dy);
        const uint32_t next = max(nd.skip, k + 1);
        if (d2 > nd.l2 * inv_theta2) {
            if ((inv_band2 == 0.f || !(d2 > nd.l2 * inv_band2)) && c < cap) pairs[(size_t)t * cap + c++] = k;
            k = next;
        } else if (nd.meta & kMetaPP) {
            k = next;
        } else {
            k = k + 1;
        }
    }
    counts[t] = c;
}

// One wave per pair (slot t, c-th cell): FP64 sum over the cell's particles (sink excluded by
// index) minus the FP64 monopole, in units of M l^2 / r^4; the sample row holds the cell's
// features and the pair's offset features w = d / r, q = l / r (d = c - p).
__global__ __launch_bounds__(kBlock) void k_label_pairs(const float4* __restrict__ pos4,
                                                        const Node* __restrict__ nodes,
                                                        const float* __restrict__ feat,
                                                        const BuildParams* __restrict__ prm,
                                                        const uint32_t* __restrict__ sinks,
                                                        const uint32_t* __restrict__ pairs,
                                                        const uint32_t* __restrict__ counts,
                                                        const uint32_t* __restrict__ offsets,
                                                        uint32_t ns, uint32_t cap, double eps2,
                                                        float* __restrict__ Xo,
                                                        float* __restrict__ To, uint32_t total) {
    const int lane = threadIdx.x & 63;
    const uint32_t gw = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (gw >= total) return;
    // find the slot whose range holds gw (offsets is an exclusive scan of counts)
    uint32_t lo = 0, hi = ns;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (offsets[mid] <= gw) lo = mid; else hi = mid;
    }
    const uint32_t t = lo, c = gw - offsets[t];
    const uint32_t sink = sinks[t];
    const uint32_t k = pairs[(size_t)t * cap + c];
    const Node nd = nodes[k];
    const float4 me = pos4[sink];
    const double px = me.x, py = me.y;
    double sx = 0.0, sy = 0.0;
    for (uint32_t j = nd.first + lane; j < nd.first + nd.count; j += 64) {
        if (j == sink) continue;
        const float4 q = pos4[j];
        const double dx = (double)q.x - px, dy = (double)q.y - py;
        const double r2 = dx * dx + dy * dy + eps2;
        const double inv = 1.0 / sqrt(r2);
        const double s = (double)q.z * inv * inv * inv;
        sx += s * dx;
        sy += s * dy;
    }
    for (int o = 32; o > 0; o >>= 1) {
        sx += __shfl_xor(sx, o, 64);
        sy += __shfl_xor(sy, o, 64);
    }
    if (lane != 0) return;
    const double dx = (double)nd.cx - px, dy = (double)nd.cy - py;
    const double r2m = dx * dx + dy * dy;
    const double invm = 1.0 / sqrt(r2m + eps2);
    const double sm = (double)nd.mass * invm * invm * invm;
    // the cell side as the walk takes it: the FP32 root side scaled by 2^-level (exact)
    const double l = ldexp((double)prm->side, -(int)(nd.meta & kMetaLevelMask));
    const double rm = sqrt(r2m);
    const double scale = (double)nd.mass * l * l / (r2m * r2m);
    float* row = Xo + (size_t)gw * kLearnSample;
#pragma unroll
    for (int q = 0; q < kMlpIn; ++q) row[q] = feat[(size_t)k * kMlpIn + q];
    row[kMlpIn] = (float)(dx / rm);
    row[kMlpIn + 1] = (float)(dy / rm);
    row[kMlpIn + 2] = (float)(l / rm);
    To[(size_t)gw * 2] = (float)((sx - sm * dx) / scale);
    To[(size_t)gw * 2 + 1] = (float)((sy - sm * dy) / scale);
}

// even (x) and odd (y) bits of a Morton prefix, compacted
__device__ __forceinline__ uint64_t compact_even(uint64_t v) {
    v &= 0x5555555555555555ull;
    v = (v | (v >> 1)) & 0x3333333333333333ull;
    v = (v | (v >> 2)) & 0x0F0F0F0F0F0F0F0Full;
    v = (v | (v >> 4)) & 0x00FF00FF00FF00FFull;
    v = (v | (v >> 8)) & 0x0000FFFF0000FFFFull;
    v = (v | (v >> 16)) & 0x00000000FFFFFFFFull;
    return v;
}

__device__ __forceinline__ double f64_of_bits(uint64_t b) { return __longlong_as_double((long long)b); }

// third moments sum m s s s about (cx, cy) over particles [f, e), `stride` threads apart from
// `t0`, kFeatLoads loads in flight per thread (pos4 is padded past n; the tail is masked)
constexpr uint32_t kFeatLoads = 4;
__device__ __forceinline__ void third_moments(const float4* __restrict__ pos4, uint32_t f,
                                              uint32_t e, uint32_t t0, uint32_t stride, float cx,
                                              float cy, float* t) {
    for (uint32_t j0 = f + t0; j0 < e; j0 += kFeatLoads * stride) {
        float4 q[kFeatLoads];
#pragma unroll
        for (uint32_t u = 0; u < kFeatLoads; ++u) q[u] = pos4[min(j0 + u * stride, e - 1)];
#pragma unroll
        for (uint32_t u = 0; u < kFeatLoads; ++u) {
            const float m = j0 + u * stride < e ? q[u].z : 0.f;
            const float x = q[u].x - cx, y = q[u].y - cy;
            const float mx = m * x, my = m * y;
            t[0] = fmaf(mx * x, x, t[0]);
            t[1] = fmaf(mx * x, y, t[1]);
            t[2] = fmaf(mx * y, y, t[2]);
            t[3] = fmaf(my * y, y, t[3]);
        }
    }
}

// wave-aggregated append of the lanes with `want` set to list[1 + ...] (list[0] counts)
__device__ __forceinline__ void list_append(uint32_t* __restrict__ list, uint32_t cap, bool want,
                                            uint32_t v) {
    const uint64_t m = __ballot(want);
    if (!m) return;
    const int lane = threadIdx.x & 63;
    const int leader = __builtin_ctzll(m);
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(&list[0], (uint32_t)__popcll(m));
    base = __shfl(base, leader, kWave);
    const uint32_t slot = base + (uint32_t)__popcll(m & lane_mask_lt());
    if (want && slot < cap) list[1 + slot] = v;
}

__device__ __forceinline__ float cell_side_f(const BuildParams* __restrict__ prm, uint32_t meta) {
    return (float)ldexp(f64_of_bits(prm->side64), -(int)(meta & kMetaLevelMask));
}

// One thread per node: the cell features (see bh_mlp.h). Second moments come from the upward
// pass (m2); third moments are summed about the node's centre of mass over its particles, here
// for cells of at most kFeatThread particles; larger cells are listed for one wave each
// (k_cell_t3_wave, up to kFeatWave particles) or one block each (k_cell_t3_big, up to
// kLearnT3Max). The box centre follows from the Morton prefix of the node's first particle (B
// code bits per axis) and the root square, in FP64.
constexpr uint32_t kFeatThread = 64;
constexpr uint32_t kFeatWave = 2048;
template <typename K>
__global__ __launch_bounds__(kBlock) void k_cell_features(const float4* __restrict__ pos4,
                                                          const Node* __restrict__ nodes,
                                                          const float4* __restrict__ m2,
                                                          const K* __restrict__ codes, int B,
                                                          const BuildParams* __restrict__ prm,
                                                          uint32_t cap_nodes,
                                                          float* __restrict__ feat,
                                                          uint32_t* __restrict__ wlist,
                                                          uint32_t wcap,
                                                          uint32_t* __restrict__ blist,
                                                          uint32_t bcap) {
    const uint32_t nn = min(prm->n_nodes, cap_nodes);
    if (blockIdx.x * kBlock >= nn) return;  // whole block
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    const bool live = k < nn;
    const Node nd = nodes[live ? k : nn - 1];
    list_append(wlist, wcap, live && nd.count > kFeatThread && nd.count <= kFeatWave, k);
    list_append(blist, bcap, live && nd.count > kFeatWave && nd.count <= kLearnT3Max, k);
    if (!live) return;
    float t[4] = {0.f, 0.f, 0.f, 0.f};
    if (nd.count <= kFeatThread) third_moments(pos4, nd.first, nd.first + nd.count, 0, 1, nd.cx, nd.cy, t);
    const int L = (int)(nd.meta & kMetaLevelMask);
    const uint64_t pre = L > 0 ? (uint64_t)codes[nd.first] >> (2 * (B - L)) : 0ull;
    const double l64 = ldexp(f64_of_bits(prm->side64), -L);
    const double bx = f64_of_bits(prm->minx64) + ((double)compact_even(pre) + 0.5) * l64;
    const double by = f64_of_bits(prm->miny64) + ((double)compact_even(pre >> 1) + 0.5) * l64;
    const float l = (float)l64;
    const float4 s2 = m2[k];
    const float a = 1.0f / (nd.mass * l * l), b = a / l;
    float* o = feat + (size_t)k * kMlpIn;
    o[0] = s2.x * a;
    o[1] = s2.y * a;
    o[2] = s2.z * a;
    o[3] = t[0] * b;
    o[4] = t[1] * b;
    o[5] = t[2] * b;
    o[6] = t[3] * b;
    o[7] = (float)(((double)nd.cx - bx) / l64);
    o[8] = (float)(((double)nd.cy - by) / l64);
    o[9] = (float)(log2((double)nd.count) / 16.0);
}

// Third moments of the cells listed for one wave each (grid-stride over the list).
__global__ __launch_bounds__(kBlock) void k_cell_t3_wave(const float4* __restrict__ pos4,
                                                         const Node* __restrict__ nodes,
                                                         const BuildParams* __restrict__ prm,
                                                         const uint32_t* __restrict__ wlist,
                                                         uint32_t wcap,
                                                         float* __restrict__ feat) {
    const uint32_t nw = min(wlist[0], wcap);
    const int lane = threadIdx.x & 63;
    const uint32_t gw = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    for (uint32_t e = gw; e < nw; e += gridDim.x * kWavesPerBlock) {
        const uint32_t k = wlist[1 + e];
        const Node nd = nodes[k];
        float t[4] = {0.f, 0.f, 0.f, 0.f};
        third_moments(pos4, nd.first, nd.first + nd.count, lane, kWave, nd.cx, nd.cy, t);
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = wave_sum_f(t[i]);
        if (lane < 4) {
            const float l = cell_side_f(prm, nd.meta);
            const float b = 1.0f / (nd.mass * l * l) / l;
            const float v = lane == 0 ? t[0] : lane == 1 ? t[1] : lane == 2 ? t[2] : t[3];
            feat[(size_t)k * kMlpIn + 3 + lane] = v * b;
        }
    }
}

// Third moments of the listed large cells: one block of kBigThreads per cell (grid-stride over
// the list), reduced in a fixed order.
constexpr int kBigThreads = 1024;
__global__ __launch_bounds__(kBigThreads) void k_cell_t3_big(const float4* __restrict__ pos4,
                                                             const Node* __restrict__ nodes,
                                                             const BuildParams* __restrict__ prm,
                                                             const uint32_t* __restrict__ big,
                                                             uint32_t big_cap,
                                                             float* __restrict__ feat) {
    __shared__ float red[kBigThreads / kWave][4];
    const uint32_t nb = min(big[0], big_cap);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (uint32_t e = blockIdx.x; e < nb; e += gridDim.x) {
        const uint32_t k = big[1 + e];
        const Node nd = nodes[k];
        float t[4] = {0.f, 0.f, 0.f, 0.f};
        third_moments(pos4, nd.first, nd.first + nd.count, threadIdx.x, kBigThreads, nd.cx,
                      nd.cy, t);
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = wave_sum_f(t[i]);
        if (lane == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[w][i] = t[i];
        __syncthreads();
        if (threadIdx.x < 4) {
            float v = 0.f;
            for (int q = 0; q < kBigThreads / kWave; ++q) v += red[q][threadIdx.x];
            const float l = cell_side_f(prm, nd.meta);
            const float b = 1.0f / (nd.mass * l * l) / l;
            feat[(size_t)k * kMlpIn + 3 + threadIdx.x] = v * b;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------------------
void launch_mlp_prep(hipStream_t s, const float* params, MlpBf16* w) {
    k_mlp_prep_bf16<<<1, 64, 0, s>>>(params, w);
}
void launch_mlp_infer_bf16(hipStream_t s, const float* X, uint32_t n, const MlpBf16* w, float* Y) {
    k_mlp_infer_bf16<<<div_up_u(n, 64 * kWavesPerBlock), kBlock, 0, s>>>(X, n, w, Y);
}
void launch_mlp_forward_f32(hipStream_t s, const float* X, uint32_t n, const float* p, float* Y) {
    k_mlp_forward_f32<<<div_up_u(n, kBlock), kBlock, 0, s>>>(X, n, p, Y);
}
// At most kTrainBlocks blocks as long as a block's plain FP32 sums then run over at most
// kTrainChain tiles (1,024 samples); more samples take more blocks instead of longer sums. With 256
// blocks throughout, the gradient of 4,194,240 equal samples was off by 1.9e-4 of its largest entry, now
// 1.5e-5.
uint32_t mlp_grad_chunks(uint32_t B) {
    const uint32_t tiles = div_up_u(B, kTrainTile), chains = div_up_u(tiles, kTrainChain);
    return tiles < kTrainBlocks ? tiles : chains < kTrainBlocks ? kTrainBlocks : chains;
}
uint32_t mlp_loss_blocks(uint32_t B) {
    const uint32_t g = div_up_u(B, kTrainTile);
    return g < 4 * kTrainBlocks ? g : 4 * kTrainBlocks;
}
void launch_mlp_grad(hipStream_t s, const float* X, const float* T, const uint32_t* order,
                     uint32_t B, const float* p, double* loss_part, float* partials, int terms) {
    k_mlp_train<true><<<mlp_grad_chunks(B), kBlock, 0, s>>>(X, T, order, B, p, loss_part,
                                                            partials, terms);
}
void launch_mlp_loss(hipStream_t s, const float* X, const float* T, uint32_t B, const float* p,
                     double* loss_part, int terms) {
    k_mlp_train<false><<<mlp_loss_blocks(B), kBlock, 0, s>>>(X, T, nullptr, B, p, loss_part,
                                                             nullptr, terms);
}
void launch_mlp_adam(hipStream_t s, float* p, const float* partials, uint32_t nchunks, float* m1,
                     float* m2, float lr, int step, float* grad_out, int apply) {
    k_mlp_adam<<<div_up_u(kMlpParams, 64), 64 * kAdamGroups, 0, s>>>(
        p, partials, nchunks, m1, m2, lr, 0.9f, 0.999f, 1e-8f, step, grad_out, apply);
}
void launch_mlp_adam_grad(hipStream_t s, float* p, const float* g, float* m1, float* m2, float lr,
                          int step) {
    k_mlp_adam_grad<<<div_up_u(kMlpParams, kBlock), kBlock, 0, s>>>(p, g, m1, m2, lr, 0.9f,
                                                                    0.999f, 1e-8f, step);
}
void launch_collect_pairs(hipStream_t s, const float4* pos4, const Node* nodes,
                          const BuildParams* prm, const uint32_t* sinks, uint32_t ns,
                          float inv_theta2, float inv_band2, uint32_t cap, uint32_t* pairs,
                          uint32_t* counts) {
    k_collect_pairs<<<div_up_u(ns, kBlock), kBlock, 0, s>>>(pos4, nodes, prm, sinks, ns,
                                                            inv_theta2, inv_band2, cap, pairs,
                                                            counts);
}
void launch_label_pairs(hipStream_t s, const float4* pos4, const Node* nodes, const float* feat,
                        const BuildParams* prm, const uint32_t* sinks, const uint32_t* pairs, const uint32_t* counts,
                        const uint32_t* offsets, uint32_t ns, uint32_t cap, double eps2, float* X,
                        float* T, uint32_t total) {
    if (!total) return;
    k_label_pairs<<<div_up_u(total, kWavesPerBlock), kBlock, 0, s>>>(
        pos4, nodes, feat, prm, sinks, pairs, counts, offsets, ns, cap, eps2, X, T, total);
}
void launch_cell_features(hipStream_t s, const float4* pos4, const Node* nodes, const float4* m2,
                          const void* codes, bool wide, int B, const BuildParams* prm,
                          uint32_t cap_nodes, float* feat, uint32_t* lists, uint32_t n) {
    const uint32_t wcap = cell_list_cap(n, kFeatThread), bcap = cell_list_cap(n, kFeatWave);
    uint32_t* wlist = lists;
    uint32_t* blist = lists + 1 + wcap;
    const uint32_t g = div_up_u(cap_nodes, kBlock);
    launch_fill_u32(s, wlist, 1, 0u);
    launch_fill_u32(s, blist, 1, 0u);
    if (wide)
        k_cell_features<uint64_t><<<g, kBlock, 0, s>>>(pos4, nodes, m2, (const uint64_t*)codes, B,
                                                       prm, cap_nodes, feat, wlist, wcap, blist,
                                                       bcap);
    else
        k_cell_features<uint32_t><<<g, kBlock, 0, s>>>(pos4, nodes, m2, (const uint32_t*)codes, B,
                                                       prm, cap_nodes, feat, wlist, wcap, blist,
                                                       bcap);
    k_cell_t3_wave<<<2048, kBlock, 0, s>>>(pos4, nodes, prm, wlist, wcap, feat);
    k_cell_t3_big<<<1024, kBigThreads, 0, s>>>(pos4, nodes, prm, blist, bcap, feat);
}
// cells of more than c particles are disjoint within a level: at most n / c of them per level,
// over at most kMaxLevels + 1 levels
uint32_t cell_list_cap(uint32_t n, uint32_t c) { return (n / c + 1) * (kMaxLevels + 1); }
size_t cell_features_lists_words(uint32_t n) {
    return 2 + (size_t)cell_list_cap(n, kFeatThread) + cell_list_cap(n, kFeatWave);
}
void launch_cell_coefs(hipStream_t s, const float* feat, const Node* nodes,
                       const BuildParams* prm, uint32_t cap_nodes, const MlpBf16* w,
                       float4* coef) {
    k_cell_coefs<<<div_up_u(cap_nodes, 64 * kWavesPerBlock), kBlock, 0, s>>>(feat, nodes, prm,
                                                                            cap_nodes, w, coef);
}

}  // namespace bh
