// The projections between two attention cores (layer_bridge.hpp) where nothing is kept for a backward pass: the same chain,
// its products on the bfloat16 matrix instructions at float32 precision.
//
// A float32 number is the sum of three bfloat16 numbers to 2^-27 of itself (eight bits each, what is left rounded to
// nearest again; from 2^-99 on, below which the third part is no normal number any more and 2^-126 takes the place of
// 2^-27 of itself), so a product of two of them is nine bfloat16 products, of which the three smallest (a1 b2, a2 b1, a2 b2:
// below 2^-25 of it) are left out.  The six others, exact in float32, go through v_mfma_f32_16x16x32_bf16 into ONE float32
// accumulator, the small ones first: six roundings of the sum per 32 products where v_mfma_f32_16x16x4_f32 makes eight.
// Error of the atoms' outputs against float64 (distance-only models, batches of 24 to 300 crystals, 2-norm): 1.3 to 1.4e-7
// after one layer and 1.8 to 1.95e-7 after four; with v_mfma_f32_16x16x4_f32 1.5 to 1.6e-7 and 1.9 to 2.05e-7.
//
// What bounds it: of a float32 chain the matrix instructions (10 us per 16 rows on a compute unit, 32 cycles per 1024
// products); six bfloat16 ones take 96 cycles per 8192.  The weights, 6 bytes each in the stream instead of 4, are then the
// larger part: 1.15 MB per workgroup (D = 128, F = 512) from the L2 at about 64 bytes per cycle are 8 us, so that many rows go
// 32 to a workgroup, two workgroups per compute unit in each other's waits: 22 528 rows 57 us (float32: 91), of which 45 are
// left without the loads of weights, 42 with one product of the six, 52 without the reads of rows from LDS.  48 and 64 rows
// per workgroup (one per compute unit): 59 and 72 us.
#pragma once
#include "layer_bridge.hpp"

namespace cfh {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));

constexpr int BI_PAD = 8;         // bfloat16 numbers of padding per LDS row: rows start 16 bytes apart modulo the banks
constexpr int BI_STEPS = 4;       // steps of 32 of the reduction index per group of 128
constexpr int BI_ROW = BR_CHUNK + BI_PAD;

// ---- the weight streams --------------------------------------------------------------------------------------
// As the forward streams of layer_bridge.hpp, with steps of 16 output columns n x 32 of the reduction index k: lane (kk, col)
// holds column 16 t + col and k = 32 u + 8 kk ... + 7, three planes of 64 x 16 bytes per step.
__host__ __device__ inline int split_stream_steps(int kind, int D, int F, bool next, int feat = 0) {
    return bridge_stream_steps(kind, D, F, next, feat) / 2;
}
// (the first part stays below the largest bfloat16 number, so that no finite number gets an infinite part; an infinity leaves
// an infinite second and a NaN as the third, and every sum with it is a NaN)
constexpr float BF16_LARGEST = 3.3895313892515355e38f;
__device__ __forceinline__ void split_bf16(float v, __bf16& a, __bf16& b, __bf16& c) {
    a = (__bf16)__builtin_amdgcn_fmed3f(v, -BF16_LARGEST, BF16_LARGEST);
    const float r = v - (float)a;
    b = (__bf16)r;
    c = (__bf16)(r - (float)b);
}
// Thread `thread` of the block-th 256: eight numbers of a step.
__device__ __forceinline__ void split_stream_element(const BridgeStreams& T, int block, int thread) {
    const BridgeStream& S = T.s[bridge_stream_of(T, block)];
    const int D = T.D, F = T.F, CT = D / 128, du = D / 32;
    const int e = (block - S.block0) * 256 + thread;
    if (e >= BR_WAVES * S.steps * 64) return;
    const int lane = e & 63, step = (e >> 6) % S.steps, w = (e >> 6) / S.steps;
    const int col = lane & 15, kk = lane >> 4;
    const float* W;
    int ld = D, t, u, s = step, valid = 0x7fffffff;
    const int eu = bridge_feat_steps(T.feat) / 2;
    if (S.kind == BS_INPUTS) {
        if (s < CT * eu) { W = S.Wo; ld = valid = T.feat; t = 8 * (s / eu) + w; u = s % eu; }
        else { s -= CT * eu; W = S.Wq; t = 8 * (s / du) + w; u = s % du; }
    } else {
        const int head = CT * du, per = du + 4 * CT, chunks = (F / 128) * per;
        if (s < head) { W = S.Wo; t = 8 * (s / du) + w; u = s % du; }
        else if (s < head + chunks) {
            const int c = (s - head) / per, r = (s - head) % per;
            if (r < du) { W = S.W1; t = 8 * c + w; u = r; }
            else { W = S.W2; ld = F; t = 8 * ((r - du) / 4) + w; u = 4 * c + (r - du) % 4; }
        } else { s -= head + chunks; W = S.Wq; t = 8 * (s / du) + w; u = s % du; }
    }
    const int n = 16 * t + col, k = 32 * u + 8 * kk;
    // (rows of 16-byte aligned matrices four numbers at a time; the features' are seldom a multiple of four)
    float v[8];
    const float* const row = W + (size_t)n * ld + k;
    if (valid == 0x7fffffff && (ld & 3) == 0 && ((uintptr_t)W & 15) == 0) {
        const float4 v0 = *reinterpret_cast<const float4*>(row), v1 = *reinterpret_cast<const float4*>(row + 4);
        v[0] = v0.x; v[1] = v0.y; v[2] = v0.z; v[3] = v0.w; v[4] = v1.x; v[5] = v1.y; v[6] = v1.z; v[7] = v1.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = k + i < valid ? row[i] : 0.0f;
    }
    v8bf p[3];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        __bf16 a, b, c;
        split_bf16(v[i], a, b, c);
        p[0][i] = a; p[1][i] = b; p[2][i] = c;
    }
    v8bf* const dst = reinterpret_cast<v8bf*>(S.dst) + (size_t)(w * S.steps + step) * 192 + lane;
#pragma unroll
    for (int i = 0; i < 3; i++) dst[64 * i] = p[i];
}

// A wavefront's stream, a group (four steps, 128 of the reduction index) at a time: the group being used is in registers.
struct SplitStream {
    const v8bf* base;
    v8bf r[BI_STEPS][3];
    __device__ __forceinline__ const v8bf* group(int g) const { return base + (size_t)g * (BI_STEPS * 192); }
    __device__ __forceinline__ void start(const float* stream, int steps, int g) {
        base = reinterpret_cast<const v8bf*>(stream) + (size_t)(threadIdx.x >> 6) * steps * 192 + (threadIdx.x & 63);
        const v8bf* const p = group(g);
#pragma unroll
        for (int u = 0; u < BI_STEPS; u++)
#pragma unroll
            for (int i = 0; i < 3; i++) r[u][i] = p[u * 192 + i * 64];
    }
};
// Rows in LDS: three planes, `plane` numbers apart.  acc += rows (16 tr + col) of `arow` (this lane's first of the 128 k)
// times the group in registers; group `next` is asked for as this one is used.
template <int TR>
__device__ __forceinline__ void split_sum(SplitStream& ws, int next, const __bf16* arow, int lda, int plane, v4f_b2 (&acc)[TR]) {
    const v8bf* const p = ws.group(next);
#pragma unroll
    for (int u = 0; u < BI_STEPS; u++) {
        const v8bf w0 = ws.r[u][0], w1 = ws.r[u][1], w2 = ws.r[u][2];
#pragma unroll
        for (int i = 0; i < 3; i++) ws.r[u][i] = p[u * 192 + i * 64];
        v8bf a[TR][3];
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int i = 0; i < 3; i++) a[tr][i] = *reinterpret_cast<const v8bf*>(arow + i * plane + 16 * tr * lda + 32 * u);
        __builtin_amdgcn_sched_barrier(0);      // (the loads ahead of the products, as in bridge_steps: 22 528 rows 59.6 -> 57.3 us)
#define CFH_SPLIT_TERM(I, W)                                                                                                     \
    _Pragma("unroll") for (int tr = 0; tr < TR; tr++) acc[tr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tr][I], W, acc[tr], 0, 0, 0)
        CFH_SPLIT_TERM(2, w0);
        CFH_SPLIT_TERM(0, w2);
        CFH_SPLIT_TERM(1, w1);
        CFH_SPLIT_TERM(1, w0);
        CFH_SPLIT_TERM(0, w1);
        CFH_SPLIT_TERM(0, w0);
#undef CFH_SPLIT_TERM
    }
}
__device__ __forceinline__ void split_store(__bf16* p, int plane, float v) {
    __bf16 a, b, c;
    split_bf16(v, a, b, c);
    p[0] = a; p[plane] = b; p[2 * plane] = c;
}
// Rows of a (N, ld) matrix, ld a multiple of 4 -> LDS planes [R][ld + BI_PAD], zeros past the last row.
template <int R>
__device__ __forceinline__ void split_rows(const float* __restrict__ src, int ld, int r0, int nrows, __bf16* dst) {
    const int ldd = ld + BI_PAD, plane = R * ldd;
    for (int idx = threadIdx.x * 4; idx < R * ld; idx += 64 * BR_WAVES * 4) {
        const int m = idx / ld, c = idx - m * ld;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < nrows) v = *reinterpret_cast<const float4*>(src + (size_t)(r0 + m) * ld + c);
        const float f[4] = {v.x, v.y, v.z, v.w};
        v4bf p[3];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            __bf16 x, y, z;
            split_bf16(f[i], x, y, z);
            p[0][i] = x; p[1][i] = y; p[2][i] = z;
        }
#pragma unroll
        for (int i = 0; i < 3; i++) *reinterpret_cast<v4bf*>(dst + i * plane + m * ldd + c) = p[i];
    }
}

// ---- the stages (as in layer_bridge.hpp; groups of a stream are numbered alike) --------------------------------
// x1 into x1r (the lane's four rows of its columns) and the planes s_x1.  `then`: the group behind the stage's own.
template <int TR, int CT>
__device__ __forceinline__ void split_first_stage(const BridgeArgs& P, SplitStream& ws, int then, __bf16* s_a, __bf16* s_x1,
                                                  float (&x1r)[CT][TR][4], int r0, int nrows) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BI_PAD, R = 16 * TR, plane = R * ldx;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {      // bias and residual of this wavefront's columns: asked for ahead of the products
        const int n = 16 * (8 * ct + wave) + col;
        const float bias = P.bo ? P.bo[n] : 0.0f;
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                x1r[ct][tr][c] = bias + (m < nrows ? P.xres[(size_t)(r0 + m) * D + n] : 0.0f);
            }
    }
    split_rows<R>(P.attn, D, r0, nrows, s_a);
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        v4f_b2 acc[TR];
        bridge_zero(acc);
#pragma unroll
        for (int g = 0; g < CT; g++) {
            const int at = ct * CT + g;
            split_sum(ws, at + 1 < CT * CT ? at + 1 : then, s_a + col * ldx + 8 * kk + 128 * g, ldx, plane, acc);
        }
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                x1r[ct][tr][c] += acc[tr][c];
                split_store(s_x1 + (16 * tr + 4 * kk + c) * ldx + n, plane, x1r[ct][tr][c]);
            }
    }
    __syncthreads();
}
// A chunk of h (its groups start at g) from s_x1: fn(row, column of the chunk, value).
template <int TR, int CT, typename Fn>
__device__ __forceinline__ void split_hidden_chunk(const BridgeArgs& P, SplitStream& ws, int c0, int g, int then, const __bf16* s_x1, Fn&& fn) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BI_PAD, plane = 16 * TR * ldx;
    const float bias = P.b1 ? P.b1[BR_CHUNK * c0 + 16 * wave + col] : 0.0f;
    v4f_b2 acc[TR];
    bridge_zero(acc);
#pragma unroll
    for (int i = 0; i < CT; i++) split_sum(ws, i + 1 < CT ? g + i + 1 : then, s_x1 + col * ldx + 8 * kk + 128 * i, ldx, plane, acc);
#pragma unroll
    for (int tr = 0; tr < TR; tr++)
#pragma unroll
        for (int c = 0; c < 4; c++) fn(16 * tr + 4 * kk + c, 16 * wave + col, rectified(acc[tr][c] + bias));
}
// x2 = sums + bias + x1 into the planes s_x and, with `store`, memory.
template <int TR, int CT>
__device__ __forceinline__ void split_second_sum(const BridgeArgs& P, v4f_b2 (&acc3)[CT][TR], float (&x1r)[CT][TR][4], __bf16* s_x, int r0,
                                                 int nrows, bool store) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BI_PAD, plane = 16 * TR * ldx;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        const float bias = P.b2 ? P.b2[n] : 0.0f;
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                const float val = acc3[ct][tr][c] + bias + x1r[ct][tr][c];
                if (P.qs) split_store(s_x + m * ldx + n, plane, val);
                if (store && m < nrows) P.x2[(size_t)(r0 + m) * D + n] = val;
            }
    }
}
// The inputs of the next layer from the planes s_x, column tiles ct0 .. ct1 - 1 of this wavefront; group g0 of the stream is
// the first of ct0.  `turn`: LDS, 16 x 17 floats per wavefront.
template <int TR, int CT>
__device__ __forceinline__ void split_inputs_stage(const BridgeArgs& P, SplitStream& ws, int g0, int ct0, int ct1, const __bf16* s_x,
                                                   float* turn, int r0, int nrows) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BI_PAD, plane = 16 * TR * ldx;
    turn += wave * (16 * 17);
#pragma unroll 1
    for (int ct = ct0; ct < ct1; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        const int part = ct / CT, cc = n - part * D;          // 128 columns of a stage belong to one of query, key, value
        const float bias = P.bq ? P.bq[n] : 0.0f;
        v4f_b2 acc[TR];
        bridge_zero(acc);
#pragma unroll
        for (int g = 0; g < CT; g++) split_sum(ws, ++g0, s_x + col * ldx + 8 * kk + 128 * g, ldx, plane, acc);
        float* const dst = part == 0 ? P.qs : (part == 1 ? P.k : P.v);
        const float scale = part == 0 ? P.q_scale : 1.0f;
#pragma unroll
        for (int tr = 0; tr < TR; tr++) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                acc[tr][c] += bias;
                if (m < nrows) dst[(size_t)(r0 + m) * D + cc] = acc[tr][c] * scale;
            }
            if (part != 0) continue;
            const int hh = cc >> 4;
            wave_sync();
#pragma unroll
            for (int c = 0; c < 4; c++) turn[(4 * kk + c) * 17 + col] = acc[tr][c];
            wave_sync();
            const int m = 16 * tr + lane;
            if (lane < 16 && m < nrows) {
                float alpha = 0.0f;
#pragma unroll
                for (int d = 0; d < DH; d++) alpha = fmaf(turn[lane * 17 + d], P.lattice_w[hh * DH + d], alpha);
                if (P.gauss) alpha = (alpha + P.gauss[1]) * P.gauss[0];
                const float u = alpha * P.c1;
                const float ex = u > 0.0f ? u : expm1f(u);
                P.a[(size_t)(r0 + m) * P.H + hh] = ((1.0f - P.lb) * ex + 1.0f) * P.c2;
            }
        }
    }
}

// grid: ceil(N / (16 TR)) workgroups of 512 threads; D = 128 CT, F a multiple of 128.
template <int TR, int CT>
__global__ __launch_bounds__(64 * BR_WAVES, CT == 1 ? 4 : 2) void bridge_infer_kernel(const BridgeArgs P) {
    constexpr int D = 128 * CT, ldx = D + BI_PAD, R = 16 * TR;
    using G = BridgeGroups<CT>;
    __shared__ __attribute__((aligned(16))) __bf16 s_a[3 * R * ldx];      // attention output, later every second chunk of h
    __shared__ __attribute__((aligned(16))) __bf16 s_x1[3 * R * ldx];     // x1, later x2
    __shared__ __attribute__((aligned(16))) __bf16 s_h[3 * R * BI_ROW];   // the other chunks of h; the alpha stage at the end
    static_assert(sizeof(s_h) >= BR_WAVES * 16 * 17 * sizeof(float), "the pieces of LDS for alpha fit a chunk");
    const int lane = threadIdx.x & 63, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * R, nrows = min(R, P.N - r0);
    SplitStream ws;
    ws.start(P.stream, P.steps, 0);
    float x1r[CT][TR][4];
    v4f_b2 acc3[CT][TR];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) bridge_zero(acc3[ct]);
    split_first_stage<TR, CT>(P, ws, G::HEAD, s_a, s_x1, x1r, r0, nrows);
    const int chunks = P.F / BR_CHUNK;
#pragma unroll 1
    for (int c0 = 0; c0 < chunks; c0++) {
        __bf16* const hb = c0 & 1 ? s_a : s_h;
        const int g = G::HEAD + c0 * G::CHUNK;
        split_hidden_chunk<TR, CT>(P, ws, c0, g, g + CT, s_x1,
                                   [&](int m, int n, float val) { split_store(hb + m * BI_ROW + n, R * BI_ROW, val); });
        __syncthreads();          // (the other chunk buffer was last read before the barrier of the chunk in between)
#pragma unroll
        for (int ct = 0; ct < CT; ct++) split_sum(ws, g + CT + ct + 1, hb + col * BI_ROW + 8 * kk, BI_ROW, R * BI_ROW, acc3[ct]);
    }
    split_second_sum<TR, CT>(P, acc3, x1r, s_x1, r0, nrows, true);      // (s_x1 was last read before the last barrier)
    if (!P.qs) return;
    __syncthreads();
    split_inputs_stage<TR, CT>(P, ws, G::HEAD + chunks * G::CHUNK, 0, 3 * CT, s_x1, reinterpret_cast<float*>(s_h), r0, nrows);
}
// The same chain in two launches, for few rows.  First: x1, a chunk of h and what it adds to x2 per workgroup, grid (tiles of
// 16 rows, chunks); the parts (chunks, N, D) in P.h, the first with x1 and the bias.  (h through memory and its 512 columns
// in the second launch: 4.4 and 8.2 us for 16 rows, three quarters of the weights behind the wait; so 5.2
// and 4.0, and with float32 products 4.7 and 9.6 in a pass.)
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void bridge_infer_split1_kernel(const BridgeArgs P) {
    constexpr int D = 128 * CT, ldx = D + BI_PAD;
    using G = BridgeGroups<CT>;
    __shared__ __attribute__((aligned(16))) __bf16 s_a[3 * 16 * ldx];
    __shared__ __attribute__((aligned(16))) __bf16 s_x1[3 * 16 * ldx];
    __shared__ __attribute__((aligned(16))) __bf16 s_h[3 * 16 * BI_ROW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * 16, nrows = min(16, P.N - r0), c0 = blockIdx.y;
    const int g = G::HEAD + c0 * G::CHUNK;
    SplitStream ws;
    ws.start(P.stream, P.steps, 0);
    float x1r[CT][1][4];
    split_first_stage<1, CT>(P, ws, g, s_a, s_x1, x1r, r0, nrows);
    split_hidden_chunk<1, CT>(P, ws, c0, g, g + CT, s_x1,
                              [&](int m, int n, float val) { split_store(s_h + m * BI_ROW + n, 16 * BI_ROW, val); });
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        const float bias = c0 == 0 && P.b2 ? P.b2[n] : 0.0f;
        v4f_b2 acc[1];
        bridge_zero(acc);
        split_sum(ws, g + CT + ct + 1, s_h + col * BI_ROW + 8 * kk, BI_ROW, 16 * BI_ROW, acc);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int m = 4 * kk + c;
            if (m < nrows) P.h[((size_t)c0 * P.N + r0 + m) * D + n] = acc[0][c] + (c0 == 0 ? bias + x1r[ct][0][c] : 0.0f);
        }
    }
}
// Second: x2 and one of query, key, value per workgroup, grid (tiles, 3), or (tiles, 1) at the end of the chain.
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void bridge_infer_split2_kernel(const BridgeArgs P) {
    constexpr int D = 128 * CT, ldx = D + BI_PAD, AHEAD = 4;
    using G = BridgeGroups<CT>;
    __shared__ __attribute__((aligned(16))) __bf16 s_x[3 * 16 * ldx];
    __shared__ float s_turn[BR_WAVES * 16 * 17];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * 16, nrows = min(16, P.N - r0), part = blockIdx.y;
    const int chunks = P.F / BR_CHUNK;
    const int g4 = G::HEAD + chunks * G::CHUNK + part * CT * CT;
    SplitStream ws;
    if (P.qs) ws.start(P.stream, P.steps, g4);
    float sum[CT][4];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int c = 0; c < 4; c++) sum[ct][c] = 0.0f;
    for (int k0 = 0; k0 < chunks; k0 += AHEAD) {      // the chunks' parts in their order, four in flight
        float v[AHEAD][CT][4];
#pragma unroll
        for (int k = 0; k < AHEAD; k++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int row = r0 + min(4 * kk + c, nrows - 1);
                    v[k][ct][c] = P.h[((size_t)min(k0 + k, chunks - 1) * P.N + row) * D + 16 * (8 * ct + wave) + col];
                }
#pragma unroll
        for (int k = 0; k < AHEAD; k++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int c = 0; c < 4; c++) sum[ct][c] += k0 + k < chunks ? v[k][ct][c] : 0.0f;
    }
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int m = 4 * kk + c, n = 16 * (8 * ct + wave) + col;
            if (P.qs) split_store(s_x + m * ldx + n, 16 * ldx, sum[ct][c]);
            if (part == 0 && m < nrows) P.x2[(size_t)(r0 + m) * D + n] = sum[ct][c];
        }
    if (!P.qs) return;
    __syncthreads();
    split_inputs_stage<1, CT>(P, ws, g4, part * CT, (part + 1) * CT, s_x, s_turn, r0, nrows);
}

// The start of the chain: the atoms' embedding x0 = x We^T, x (N, feat), to x2, and the inputs of the first layer.  The rows
// of x, a few dozen columns and not 16-byte aligned, are staged word by word, zeros behind the last feature.  grid (tiles of
// 16 TR rows, query / key / value or 1: all three); dynamic LDS: the planes of 16 TR rows of x.
template <int TR, int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void front_infer_kernel(const BridgeArgs P) {
    extern __shared__ __attribute__((aligned(16))) float s_dyn[];
    constexpr int D = 128 * CT, ldx = D + BI_PAD, R = 16 * TR;
    __shared__ __attribute__((aligned(16))) __bf16 s_x[3 * R * ldx];
    __shared__ float s_turn[BR_WAVES * 16 * 17];
    __bf16* const s_f = reinterpret_cast<__bf16*>(s_dyn);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * R, nrows = min(R, P.N - r0);
    const int feat = P.feat, pad = 16 * bridge_feat_steps(feat), ldf = pad + BI_PAD, eg = pad / 128;
    const int parts = gridDim.y == 1 ? 3 : 1, part = blockIdx.y, g0 = CT * eg + part * CT * CT;
    SplitStream ws;
    ws.start(P.stream, P.steps, 0);
    // (a wavefront's rows of 128 features with all loads in flight: one by one 22 528 rows 34 us for the launch instead of 29, 8 rows 6.5 and 5.8)
    constexpr int ROWS = R / BR_WAVES;
    for (int c0 = 0; c0 < pad; c0 += 128) {
        float v[ROWS][2];
#pragma unroll
        for (int r = 0; r < ROWS; r++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int m = wave + BR_WAVES * r, c = c0 + 64 * j + lane;
                v[r][j] = P.attn[(size_t)(r0 + min(m, nrows - 1)) * feat + min(c, feat - 1)];
            }
#pragma unroll
        for (int r = 0; r < ROWS; r++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int m = wave + BR_WAVES * r, c = c0 + 64 * j + lane;
                split_store(s_f + m * ldf + c, R * ldf, m < nrows && c < feat ? v[r][j] : 0.0f);
            }
    }
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        v4f_b2 acc[TR];
        bridge_zero(acc);
#pragma unroll 1
        for (int g = 0; g < eg; g++) {
            const int at = ct * eg + g;
            split_sum(ws, at + 1 < CT * eg ? at + 1 : g0, s_f + col * ldf + 8 * kk + 128 * g, ldf, R * ldf, acc);
        }
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                split_store(s_x + m * ldx + n, R * ldx, acc[tr][c]);
                if (part == 0 && m < nrows) P.x2[(size_t)(r0 + m) * D + n] = acc[tr][c];
            }
    }
    __syncthreads();
    split_inputs_stage<TR, CT>(P, ws, g0, part * CT, (part + parts) * CT, s_x, s_turn, r0, nrows);
}

}  // namespace cfh
