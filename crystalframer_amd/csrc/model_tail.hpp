// What follows the encoder: the mean over the atoms of every crystal and a head of linear layers (the reference's
// pooling and mlp, models/pooling.py:19-25, models/latticeformer.py:150-207), one launch each way.  A few thousand
// rows of a few hundred floats: a launch per layer is all latency (5 to 7 us each for 256 crystals, 1.5 us of it work).
// A workgroup takes up to 16 crystals -- the M of v_mfma_f32_16x16x4 -- through the chain with the rows in LDS.
#pragma once
#include "device_common.hpp"

namespace cfh {

typedef float v4f_t __attribute__((ext_vector_type(4)));

constexpr int TAIL_ROWS = 16;
constexpr int TAIL_WAVES = 8;
constexpr int TAIL_PAD = 4;
constexpr int TAIL_MAX_LINEARS = 6;

struct TailLinear {
    const float* W; const float* b;      // (O, K), (O)
    float* y;                            // forward: (B, O) result (with the rectifier applied)
    float* gy;                           // backward: (B, O) gradient of the result before the rectifier; the last one is given
    int K, O, relu;
};
struct TailArgs {
    const float* x;                      // (N, D)
    const int64_t* atom_start;           // (B + 1)
    float* pooled;                       // (B, D)
    float* gx;                           // (N, D) backward: gradient of x, every atom its crystal's over their number
    TailLinear lin[TAIL_MAX_LINEARS];
    int B, D, per_wg, nlin, ld;          // ld: floats of an LDS row (the widest row rounded up to 4, + TAIL_PAD)
};

// Dynamic LDS: 2 x 16 rows of ld floats.
// per_wg crystals per workgroup: one for small batches (a crystal of 200 atoms is 100 KB to add up, and the chip has
// 256 compute units to do it), 16 for thousands of crystals (the weights are read once per workgroup).
__global__ __launch_bounds__(64 * TAIL_WAVES) void model_tail_fwd_kernel(const TailArgs P) {
    extern __shared__ __attribute__((aligned(16))) float tail_lds[];
    __shared__ float4 part[64 * TAIL_WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int b0 = blockIdx.x * P.per_wg, nrows = min(P.per_wg, P.B - b0);
    const int ld = P.ld, D = P.D, Q = D >> 2;
    float* in = tail_lds;
    float* outb = tail_lds + TAIL_ROWS * ld;
    for (int u = threadIdx.x; u < TAIL_ROWS * ld; u += 64 * TAIL_WAVES) in[u] = 0.0f;
    // mean over the atoms: Q threads per row, R rows at a time, S of them on one crystal, added up in a fixed order
    // (S as in crystal_mean_fwd_vec_kernel: the same sums to the last bit)
    const int R = (64 * TAIL_WAVES) / Q, S = min(R, max(1, 256 / Q)), at_once = R / S;
    const int rr = (int)threadIdx.x / Q, q = (int)threadIdx.x - rr * Q;
    const float4* const x4 = reinterpret_cast<const float4*>(P.x);
    __syncthreads();
    for (int c0 = 0; c0 < nrows; c0 += at_once) {
        const int c = c0 + rr / S, sl = rr % S;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        const bool live = rr < at_once * S && c < nrows;
        int64_t s = 0, t = 0;
        if (live) {
            s = P.atom_start[b0 + c]; t = P.atom_start[b0 + c + 1];
            for (int64_t i = s + sl; i < t; i += S) {
                const float4 v = x4[(size_t)i * Q + q];
                acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
            }
        }
        part[threadIdx.x] = acc;
        __syncthreads();
        if (live && sl == 0) {
            for (int k = 1; k < S; k++) {
                const float4 v = part[threadIdx.x + k * Q];
                acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
            }
            const float inv = t > s ? 1.0f / (float)(t - s) : 0.0f;
            const float4 m = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
            *reinterpret_cast<float4*>(in + c * ld + 4 * q) = m;
            reinterpret_cast<float4*>(P.pooled)[(size_t)(b0 + c) * Q + q] = m;
        }
        __syncthreads();
    }
    for (int li = 0; li < P.nlin; li++) {
        const TailLinear& T = P.lin[li];
        const int K = T.K, O = T.O;
        for (int t = wave; 16 * t < O; t += TAIL_WAVES) {
            const int n = 16 * t + col, nc = min(n, O - 1);
            const float* const wrow = T.W + (size_t)nc * K + 4 * kk;
            const float* const arow = in + col * ld + 4 * kk;
            v4f_t acc = {0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < K; k0 += 128) {
                float4 w4[8];
#pragma unroll
                for (int u = 0; u < 8; u++) w4[u] = *reinterpret_cast<const float4*>(wrow + min(k0 + 16 * u, K - 16));
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    if (k0 + 16 * u >= K) break;
                    const float4 a4 = *reinterpret_cast<const float4*>(arow + k0 + 16 * u);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.x, w4[u].x, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.y, w4[u].y, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.z, w4[u].z, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.w, w4[u].w, acc, 0, 0, 0);
                }
            }
            const float bias = T.b ? T.b[nc] : 0.0f;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 4 * kk + c;
                float val = acc[c] + bias;
                if (T.relu) val = rectified(val);
                if (n < O) {
                    outb[m * ld + n] = val;
                    if (m < nrows) T.y[(size_t)(b0 + m) * O + n] = val;
                }
            }
        }
        __syncthreads();
        float* const tmp = in; in = outb; outb = tmp;
    }
}

// Gradients of the head's inputs: gy of the last layer is given (its rectifier, if it has one, is applied here and the
// result written to gy), the others and the atoms' are made here.  Dynamic LDS as in the forward kernel.
__global__ __launch_bounds__(64 * TAIL_WAVES) void model_tail_bwd_kernel(const TailArgs P, const float* __restrict__ gout) {
    extern __shared__ __attribute__((aligned(16))) float tail_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int b0 = blockIdx.x * P.per_wg, nrows = min(P.per_wg, P.B - b0);
    const int ld = P.ld;
    float* g = tail_lds;
    float* gin = tail_lds + TAIL_ROWS * ld;
    for (int u = threadIdx.x; u < 2 * TAIL_ROWS * ld; u += 64 * TAIL_WAVES) tail_lds[u] = 0.0f;
    __syncthreads();
    {
        const TailLinear& T = P.lin[P.nlin - 1];
        for (int u = threadIdx.x; u < nrows * T.O; u += 64 * TAIL_WAVES) {
            const int m = u / T.O, n = u - m * T.O;
            const size_t at = (size_t)(b0 + m) * T.O + n;
            float v = gout[at];
            if (T.relu && !(T.y[at] > 0.0f)) v = 0.0f;
            g[m * ld + n] = v;
            T.gy[at] = v;
        }
    }
    __syncthreads();
    for (int li = P.nlin - 1; li >= 0; li--) {
        const TailLinear& T = P.lin[li];
        const int K = T.K, O = T.O, steps = (O + 3) / 4;
        const bool mask = li > 0 && P.lin[li > 0 ? li - 1 : 0].relu;
        const float* const ymask = li > 0 ? P.lin[li - 1].y : nullptr;
        float* const dst = li > 0 ? P.lin[li - 1].gy : nullptr;
        for (int t = wave; 16 * t < K; t += TAIL_WAVES) {
            const int n = 16 * t + col;                       // (K is a multiple of 16)
            v4f_t acc = {0.f, 0.f, 0.f, 0.f};
            for (int s0 = 0; s0 < steps; s0 += 8) {
                float w[8];
                int o[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    // (whole chunks of 16 in the order of small_linear_dx_kernel, which steps through a lane's four
                    // consecutive features: the same sums to the last bit)
                    o[u] = O % 16 == 0 ? 16 * ((s0 + u) >> 2) + 4 * kk + ((s0 + u) & 3) : 4 * (s0 + u) + kk;
                    w[u] = T.W[(size_t)min(o[u], O - 1) * K + n];
                }
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    if (s0 + u >= steps) break;
                    const float a = o[u] < O ? g[col * ld + o[u]] : 0.0f;
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, w[u], acc, 0, 0, 0);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 4 * kk + c;
                float v = acc[c];
                if (m < nrows) {
                    if (mask && !(ymask[(size_t)(b0 + m) * K + n] > 0.0f)) v = 0.0f;
                    if (dst) dst[(size_t)(b0 + m) * K + n] = v;
                }
                gin[m * ld + n] = v;
            }
        }
        __syncthreads();
        float* const tmp = g; g = gin; gin = tmp;
    }
    // the mean over the atoms: Q threads per atom
    const int Q = P.D >> 2, R = (64 * TAIL_WAVES) / Q;
    const int rr = (int)threadIdx.x / Q, q = (int)threadIdx.x - rr * Q;
    if (rr >= R) return;
    for (int c = 0; c < nrows; c++) {
        const int64_t s = P.atom_start[b0 + c], t = P.atom_start[b0 + c + 1];
        const float inv = 1.0f / (float)(t - s);
        float4 v = *reinterpret_cast<const float4*>(g + c * ld + 4 * q);
        v.x *= inv; v.y *= inv; v.z *= inv; v.w *= inv;
        for (int64_t i = s + rr; i < t; i += R) reinterpret_cast<float4*>(P.gx)[(size_t)i * Q + q] = v;
    }
}

}  // namespace cfh
