// The projections between the attention cores of two consecutive encoder layers, which act on every atom (row)
// separately, in one launch each way (two for few rows):
//     x1  = x_res + attn Wo^T + bo              (output projection of the attention + residual)
//     h   = relu(x1 W1^T + b1)                  (feed-forward, first half)
//     x2  = x1 + h W2^T + b2                    (second half + residual: the layer's output)
//     qkv = x2 Wqkv^T + bqkv                    (stacked input projection of the NEXT layer, optional)
//     qs, k, v, a = split / scaled query / Gaussian coefficient of qkv (see attention_inputs.hpp)
// and their input gradients
//     gqkv from the gradients of qs, k, v, a;  g2 = g_x2 + gqkv Wqkv;  gh = (g2 W2) [h > 0];  g1 = g2 + gh W1;  g_attn = g1 Wo.
// The reference runs them as separate framework calls (models/indexed_lattice_multi_head_attention_cuda.py:
// 399-409 and the out_proj behind :734, models/indexed_latticeformer_encoder.py:606-648 with post-norm
// switched off).  A workgroup of eight wavefronts takes 16 TR rows -- TR times the M of v_mfma_f32_16x16x4 -- through
// the whole chain with the activations in LDS; the wavefronts share a stage's output columns, 16 at a time.
//
// What bounds it: a workgroup has 3072 TR of the 32-cycle matrix instructions (10 us on a compute unit's four SIMDs) and
// 768 KB of weights to read from the L2.  Read from the matrices as they are, a lane's four consecutive k of its row are
// 64 cache lines per load instruction, twice the time of the products; turned in LDS on the way, with the loads one batch
// ahead and a trip to the L2 at the head of every stage, the chain took 22 us for one crystal, 28 us at 2372 atoms and
// 138 us at 22 528.  One launch per product (four instead of one, more compute units per row) came to 17, 30 and 133 us:
// each launch waits for what the one before it wrote.  So the weights are laid out once per pass in the order in which
// the wavefronts use them (bridge_stream_kernel): every wavefront then reads ONE contiguous stream, 1 KB per load
// instruction, eight instructions ahead, on through the stages and the barriers between them.
#pragma once
#include "attention_inputs.hpp"
#include "device_common.hpp"

namespace cfh {

typedef float v4f_b2 __attribute__((ext_vector_type(4)));

constexpr int BR_WAVES = 8;
constexpr int BR_PAD = 4;         // floats of padding per LDS row
constexpr int BR_RING = 8;        // steps of the weight stream in flight
constexpr int BR_CHUNK = 16 * BR_WAVES;      // columns of the feed-forward block's inside that are in LDS at a time

// ---- the weight streams --------------------------------------------------------------------------------------
// A step is what one wavefront multiplies at once: 16 output columns n x 16 of the reduction index k, 64 lanes x 4 floats;
// lane (kk, col) holds column 16 t + col and k = 16 u + 4 kk ... + 3.  Stream of a wavefront w (D = 128 CT, tiles of a
// stage t = 8 ct + w):
//   forward    Wo: ct < CT, u < D/16;  per chunk c of 128 columns of F: W1 tile 8 c + w, u < D/16, then W2: ct < CT, the
//              chunk's 8 u;  with a next layer Wqkv: ct < 3 CT, u < D/16
//   backward   (the same matrices from the other side) with a next layer Wqkv: ct < CT, u < 3D/16;  per chunk: W2 tile
//              8 c + w, u < D/16, then W1: ct < CT, the chunk's 8 u;  Wo: ct < CT, u < D/16
//   inputs     (first layer) forward: the embedding We (D, feat), ct < CT, u < E = feat / 16 rounded up to a multiple of 8
//              (zeros past the last feature), then Wqkv: ct < 3 CT, u < D/16;  backward Wqkv: ct < CT, u < 3D/16
enum { BS_FORWARD = 0, BS_BACKWARD = 1, BS_INPUTS = 2, BS_INPUTS_BACKWARD = 3 };
__host__ __device__ inline int bridge_feat_steps(int feat) { return (feat + 127) / 128 * 8; }
__host__ __device__ inline int bridge_stream_steps(int kind, int D, int F, bool next, int feat = 0) {
    const int CT = D / 128, du = D / 16, q = 3 * CT * du;
    if (kind >= BS_INPUTS) return q + (kind == BS_INPUTS ? CT * bridge_feat_steps(feat) : 0);
    return CT * du + (F / 128) * (du + 8 * CT) + (next ? q : 0);
}
struct BridgeStream {
    const float* Wo; const float* W1; const float* W2; const float* Wq;      // (D, D), (F, D), (D, F), (3 D, D) or null;
                                  // inputs: Wo the embedding (D, feat)
    float* dst;                   // BR_WAVES x steps x 64 float4
    int kind, steps, block0;
};
constexpr int BR_MAX_STREAMS = 24;
struct BridgeStreams {
    BridgeStream s[BR_MAX_STREAMS];
    int first[BR_MAX_STREAMS];    // their block0
    int n, D, F, feat;
    int split;                    // see bridge_infer.hpp
};
// The stream that a block (the same in all lanes) belongs to: the first blocks lie side by side and come with a load or two,
// where a scan of the streams waited for the arguments' memory once per stream.
__device__ __forceinline__ int bridge_stream_of(const BridgeStreams& T, int block) {
    const int b = __builtin_amdgcn_readfirstlane(block);
    int si = 0;
#pragma unroll
    for (int k = 1; k < BR_MAX_STREAMS; k++) si += k < T.n && b >= T.first[k] ? 1 : 0;
    return si;
}
// A thread per float4 of the streams: thread `thread` of the block-th 256.
__device__ __forceinline__ void bridge_stream_element(const BridgeStreams& T, int block, int thread) {
    const BridgeStream& S = T.s[bridge_stream_of(T, block)];
    const int D = T.D, F = T.F, CT = D / 128, du = D / 16;
    const int e = (block - S.block0) * 256 + thread;
    if (e >= BR_WAVES * S.steps * 64) return;
    const int lane = e & 63, step = (e >> 6) % S.steps, w = (e >> 6) / S.steps;
    const int col = lane & 15, kk = lane >> 4;
    const bool back = S.kind == BS_BACKWARD || S.kind == BS_INPUTS_BACKWARD;
    // which matrix, tile and u
    const float* W = nullptr;
    int ld = D, t = 0, u = 0, s = step;
    if (S.kind == BS_INPUTS) {
        const int eu = bridge_feat_steps(T.feat);
        if (s < CT * eu) {
            const int n = 16 * (8 * (s / eu) + w) + col, k = 16 * (s % eu) + 4 * kk;
            float4 v;
            v.x = k + 0 < T.feat ? S.Wo[(size_t)n * T.feat + k + 0] : 0.0f;
            v.y = k + 1 < T.feat ? S.Wo[(size_t)n * T.feat + k + 1] : 0.0f;
            v.z = k + 2 < T.feat ? S.Wo[(size_t)n * T.feat + k + 2] : 0.0f;
            v.w = k + 3 < T.feat ? S.Wo[(size_t)n * T.feat + k + 3] : 0.0f;
            reinterpret_cast<float4*>(S.dst)[e] = v;
            return;
        }
        s -= CT * eu;
        W = S.Wq; t = 8 * (s / du) + w; u = s % du;
    }
    else if (S.kind == BS_INPUTS_BACKWARD) { W = S.Wq; t = 8 * (s / (3 * du)) + w; u = s % (3 * du); }
    else {
        const int head = back ? (S.Wq ? CT * 3 * du : 0) : CT * du;          // steps before the chunks
        const int per = du + 8 * CT, chunks = (F / 128) * per;
        if (s < head) {
            if (back) { W = S.Wq; t = 8 * (s / (3 * du)) + w; u = s % (3 * du); }
            else { W = S.Wo; t = 8 * (s / du) + w; u = s % du; }
        } else if (s < head + chunks) {
            const int c = (s - head) / per, r = (s - head) % per;
            if (r < du) { W = back ? S.W2 : S.W1; ld = back ? F : D; t = 8 * c + w; u = r; }
            else { W = back ? S.W1 : S.W2; ld = back ? D : F; t = 8 * ((r - du) / 8) + w; u = 8 * c + (r - du) % 8; }
        } else {
            s -= head + chunks;
            W = back ? S.Wo : S.Wq; t = 8 * (s / du) + w; u = s % du;
        }
    }
    const int n = 16 * t + col, k = 16 * u + 4 * kk;
    float4 v;
    if (back) {                   // the operand is W[k][n]
        v.x = W[(size_t)(k + 0) * ld + n]; v.y = W[(size_t)(k + 1) * ld + n];
        v.z = W[(size_t)(k + 2) * ld + n]; v.w = W[(size_t)(k + 3) * ld + n];
    } else {
        v = *reinterpret_cast<const float4*>(W + (size_t)n * ld + k);
    }
    reinterpret_cast<float4*>(S.dst)[e] = v;
}

// grid: blocks of all streams, 256 threads.
__global__ __launch_bounds__(256) void bridge_stream_kernel(const BridgeStreams T) {
    bridge_stream_element(T, (int)blockIdx.x, (int)threadIdx.x);
}

// A wavefront's stream, eight steps (a group) at a time: the group being used is in registers.
struct WeightStream {
    const v4f_b2* base;           // this lane's place in the stream
    v4f_b2 r[BR_RING];
    __device__ __forceinline__ const v4f_b2* group(int g) const { return base + (size_t)g * (BR_RING * 64); }
    __device__ __forceinline__ void start(const float* stream, int steps, int g) {
        base = reinterpret_cast<const v4f_b2*>(stream) + (size_t)(threadIdx.x >> 6) * steps * 64 + (threadIdx.x & 63);
        const v4f_b2* const p = group(g);
#pragma unroll
        for (int i = 0; i < BR_RING; i++) r[i] = p[i * 64];
    }
};
// One group: acc += rows (16 tr + col) of `arow` (LDS, this lane's first float of the 128 k) times the stream.  Group
// `next` is asked for as this one is used (behind the end of a stream lies one more).  FOLD: the sum over k is made in
// slices of klen that are added up in order.
template <int TR, bool FOLD>
__device__ __forceinline__ void bridge_steps(WeightStream& ws, int next, const float* arow, int lda, v4f_b2 (&acc)[TR],
                                             v4f_b2 (&sum)[TR], int klen, int& in_slice, bool& first) {
    const v4f_b2* const p = ws.group(next);
    v4f_b2 an[TR];
#pragma unroll
    for (int tr = 0; tr < TR; tr++) an[tr] = *reinterpret_cast<const v4f_b2*>(arow + 16 * tr * lda);
#pragma unroll
    for (int u = 0; u < BR_RING; u++) {
        const v4f_b2 w = ws.r[u];
        ws.r[u] = p[u * 64];
        v4f_b2 a[TR];
#pragma unroll
        for (int tr = 0; tr < TR; tr++) {
            a[tr] = an[tr];
            if (u + 1 < BR_RING) an[tr] = *reinterpret_cast<const v4f_b2*>(arow + 16 * tr * lda + 16 * (u + 1));
        }
        // (said so, or the compiler puts the eight loads of the next group behind the products of this one, and every step's
        // rows right in front of its products: 2372 rows 21.8 -> 20.4 us forward, 25.1 -> 24.6 backward)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int tr = 0; tr < TR; tr++)
                acc[tr] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tr][j], w[j], acc[tr], 0, 0, 0);
        if (FOLD) {
            in_slice += 16;
            if (in_slice == klen) {
#pragma unroll
                for (int tr = 0; tr < TR; tr++) {
                    if (first) sum[tr] = acc[tr];
                    else sum[tr] += acc[tr];
                    acc[tr] = v4f_b2{0.f, 0.f, 0.f, 0.f};
                }
                in_slice = 0;
                first = false;
            }
        }
    }
}
template <int TR>
__device__ __forceinline__ void bridge_sum(WeightStream& ws, int next, const float* arow, int lda, v4f_b2 (&acc)[TR]) {
    int slice = 0;
    bool first = true;
    bridge_steps<TR, false>(ws, next, arow, lda, acc, acc, 0, slice, first);
}
// Groups of a stream: forward  CT^2 of Wo, per chunk CT of W1 and CT of W2, 3 CT^2 of Wqkv.
template <int CT>
struct BridgeGroups {
    static constexpr int HEAD = CT * CT, CHUNK = 2 * CT;
};
template <int TR>
__device__ __forceinline__ void bridge_zero(v4f_b2 (&acc)[TR]) {
#pragma unroll
    for (int tr = 0; tr < TR; tr++) acc[tr] = v4f_b2{0.f, 0.f, 0.f, 0.f};
}

struct BridgeArgs {
    const float* attn; const float* xres;         // (N, D); first layer: (N, feat) features, null
    const float* bo; const float* b1; const float* b2; const float* bq;      // may be null
    const float* stream; int steps;
    const float* lattice_w; const float* gauss;   // (D); device {scale, shift} or null
    float* x1; float* h; float* x2; float* qkv;   // (N, D), (N, F), (N, D), (N, 3 D); x1, h, qkv null: not written
    float* qs; float* k; float* v; float* a;      // (N, D) x 3, (N, H); null: the chain ends with x2
    int N, D, F, H, feat;
    float c1, lb, c2, q_scale;
};
// rows of a (N, ld) matrix -> LDS [16 TR][ld + BR_PAD], zeros past the last row
template <int TR>
__device__ __forceinline__ void bridge_rows(const float* __restrict__ src, int ld, int r0, int nrows, float* dst) {
    for (int idx = threadIdx.x * 4; idx < 16 * TR * ld; idx += 64 * BR_WAVES * 4) {
        const int m = idx / ld, c = idx - m * ld;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < nrows) v = *reinterpret_cast<const float4*>(src + (size_t)(r0 + m) * ld + c);
        *reinterpret_cast<float4*>(dst + m * (ld + BR_PAD) + c) = v;
    }
}
// The last stage: the inputs of the next layer from the rows s_x (LDS), column tiles ct0 .. ct1 - 1 of this wavefront;
// group g0 of the stream is the first of ct0.  `turn`: LDS, 16 x 17 floats per wavefront.  TREE: alpha as a row sum over
// the 16 lanes of a head, as attention_inputs_fwd_kernel makes it (the first layer), else its channels one after the other.
template <int TR, int CT, bool TREE>
__device__ __forceinline__ void bridge_inputs_stage(const BridgeArgs& P, WeightStream& ws, int g0, int ct0, int ct1,
                                                    const float* s_x, float* turn, int r0, int nrows) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD;
    turn += wave * (16 * 17);
#pragma unroll 1
    for (int ct = ct0; ct < ct1; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        const int part = ct / CT, cc = n - part * D;          // 128 columns of a stage belong to one of query, key, value
        const float bias = P.bq ? P.bq[n] : 0.0f;
        const float lw = part == 0 ? P.lattice_w[cc] : 0.0f;
        v4f_b2 acc[TR];
        bridge_zero(acc);
#pragma unroll
        for (int g = 0; g < CT; g++) bridge_sum(ws, ++g0, s_x + col * ldx + 4 * kk + 128 * g, ldx, acc);
        float* const dst = part == 0 ? P.qs : (part == 1 ? P.k : P.v);
        const float scale = part == 0 ? P.q_scale : 1.0f;
        auto coefficient = [&](float alpha) {
            if (P.gauss) alpha = (alpha + P.gauss[1]) * P.gauss[0];
            const float u = alpha * P.c1;
            const float ex = u > 0.0f ? u : expm1f(u);
            return ((1.0f - P.lb) * ex + 1.0f) * P.c2;
        };
#pragma unroll
        for (int tr = 0; tr < TR; tr++) {
            float val[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                val[c] = acc[tr][c] + bias;
                if (m < nrows) {
                    if (P.qkv) P.qkv[(size_t)(r0 + m) * (3 * D) + n] = val[c];
                    dst[(size_t)(r0 + m) * D + cc] = val[c] * scale;
                }
            }
            if (part != 0) continue;
            const int hh = cc >> 4;
            if (TREE) {
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int m = 16 * tr + 4 * kk + c;
                    const float co = coefficient(head_dot(m < nrows ? val[c] : 0.0f, lw));
                    if (col == 0 && m < nrows) P.a[(size_t)(r0 + m) * P.H + hh] = co;
                }
            } else {
                wave_sync();
#pragma unroll
                for (int c = 0; c < 4; c++) turn[(4 * kk + c) * 17 + col] = val[c];
                wave_sync();
                const int m = 16 * tr + lane;
                if (lane < 16 && m < nrows) {
                    float alpha = 0.0f;
#pragma unroll
                    for (int d = 0; d < DH; d++) alpha = fmaf(turn[lane * 17 + d], P.lattice_w[hh * DH + d], alpha);
                    P.a[(size_t)(r0 + m) * P.H + hh] = coefficient(alpha);
                }
            }
        }
    }
}
// First stage: x1 into s_x1 and, with `store`, memory.  `then`: the group behind the stage's own.
template <int TR, int CT>
__device__ __forceinline__ void bridge_first_stage(const BridgeArgs& P, WeightStream& ws, int then, float* s_x, float* s_x1, int r0,
                                                   int nrows, bool store) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD;
    // bias and residual of this wavefront's columns: asked for ahead of the products
    float add[CT][TR][4];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        const float bias = P.bo ? P.bo[n] : 0.0f;
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                add[ct][tr][c] = bias + (m < nrows ? P.xres[(size_t)(r0 + m) * D + n] : 0.0f);
            }
    }
    bridge_rows<TR>(P.attn, D, r0, nrows, s_x);
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        v4f_b2 acc[TR];
        bridge_zero(acc);
#pragma unroll
        for (int g = 0; g < CT; g++) {
            const int at = ct * CT + g;
            bridge_sum(ws, at + 1 < CT * CT ? at + 1 : then, s_x + col * ldx + 4 * kk + 128 * g, ldx, acc);
        }
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                const float val = acc[tr][c] + add[ct][tr][c];
                s_x1[m * ldx + n] = val;
                if (store && m < nrows) P.x1[(size_t)(r0 + m) * D + n] = val;
            }
    }
    __syncthreads();
}
// Chunk c0 of h (its groups start at g) from s_x1, into hb (LDS) if given and to memory if wanted; `then`: the group behind.
template <int TR, int CT>
__device__ __forceinline__ void bridge_hidden_chunk(const BridgeArgs& P, WeightStream& ws, int c0, int g, int then, const float* s_x1,
                                                    float* hb, int r0, int nrows) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD, ldh = BR_CHUNK + BR_PAD;
    const int n = BR_CHUNK * c0 + 16 * wave + col;
    const float bias = P.b1 ? P.b1[n] : 0.0f;
    v4f_b2 acc[TR];
    bridge_zero(acc);
#pragma unroll
    for (int i = 0; i < CT; i++) bridge_sum(ws, i + 1 < CT ? g + i + 1 : then, s_x1 + col * ldx + 4 * kk + 128 * i, ldx, acc);
#pragma unroll
    for (int tr = 0; tr < TR; tr++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int m = 16 * tr + 4 * kk + c;
            const float val = rectified(acc[tr][c] + bias);
            if (hb) hb[m * ldh + 16 * wave + col] = val;
            if (P.h && m < nrows) P.h[(size_t)(r0 + m) * P.F + n] = val;
        }
}
// x2 = sums + bias + x1 (in place in s_x1) into s_x and, with `store`, memory.
template <int TR, int CT>
__device__ __forceinline__ void bridge_second_sum(const BridgeArgs& P, v4f_b2 (&acc3)[CT][TR], const float* s_x1, float* s_x, int r0,
                                                  int nrows, bool store) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        const float bias = P.b2 ? P.b2[n] : 0.0f;
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                const float val = acc3[ct][tr][c] + bias + s_x1[m * ldx + n];
                s_x[m * ldx + n] = val;
                if (store && m < nrows) P.x2[(size_t)(r0 + m) * D + n] = val;
            }
    }
}

// grid: ceil(N / (16 TR)) workgroups of 512 threads; D = 128 CT, F a multiple of 128.
template <int TR, int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void layer_bridge_fwd_kernel(const BridgeArgs P) {
    constexpr int D = 128 * CT, ldx = D + BR_PAD, ldh = BR_CHUNK + BR_PAD, R = 16 * TR;
    using G = BridgeGroups<CT>;
    __shared__ __attribute__((aligned(16))) float s_x[R * ldx];           // attention output, later x2
    __shared__ __attribute__((aligned(16))) float s_x1[R * ldx];
    __shared__ __attribute__((aligned(16))) float s_h[2][R * ldh];        // a chunk of h; the alpha stage at the end
    static_assert(2 * R * ldh >= BR_WAVES * 16 * 17, "the pieces of LDS for alpha fit the chunks");
    const int lane = threadIdx.x & 63, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * R, nrows = min(R, P.N - r0);
    WeightStream ws;
    ws.start(P.stream, P.steps, 0);
    v4f_b2 acc3[CT][TR];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) bridge_zero(acc3[ct]);
    bridge_first_stage<TR, CT>(P, ws, G::HEAD, s_x, s_x1, r0, nrows, P.x1 != nullptr);
    const int chunks = P.F / BR_CHUNK;
#pragma unroll 1
    for (int c0 = 0; c0 < chunks; c0++) {
        float* const hb = s_h[c0 & 1];
        const int g = G::HEAD + c0 * G::CHUNK;
        bridge_hidden_chunk<TR, CT>(P, ws, c0, g, g + CT, s_x1, hb, r0, nrows);
        __syncthreads();          // (the other chunk buffer was last read before the barrier of the chunk in between)
#pragma unroll
        for (int ct = 0; ct < CT; ct++) bridge_sum(ws, g + CT + ct + 1, hb + col * ldh + 4 * kk, ldh, acc3[ct]);
    }
    bridge_second_sum<TR, CT>(P, acc3, s_x1, s_x, r0, nrows, true);
    if (!P.qs) return;
    __syncthreads();
    bridge_inputs_stage<TR, CT, false>(P, ws, G::HEAD + chunks * G::CHUNK, 0, 3 * CT, s_x, s_h[0], r0, nrows);
}
// The same chain in two launches, for few rows.  First: x1 and one chunk of h per workgroup, grid (tiles of 16 rows, chunks);
// x1 and h are kept in memory.
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void layer_bridge_fwd_split1_kernel(const BridgeArgs P) {
    constexpr int ldx = 128 * CT + BR_PAD;
    using G = BridgeGroups<CT>;
    __shared__ __attribute__((aligned(16))) float s_x[16 * ldx];
    __shared__ __attribute__((aligned(16))) float s_x1[16 * ldx];
    const int r0 = blockIdx.x * 16, nrows = min(16, P.N - r0), c0 = blockIdx.y;
    const int g = G::HEAD + c0 * G::CHUNK;
    WeightStream ws;
    ws.start(P.stream, P.steps, 0);
    bridge_first_stage<1, CT>(P, ws, g, s_x, s_x1, r0, nrows, c0 == 0);
    bridge_hidden_chunk<1, CT>(P, ws, c0, g, g, s_x1, nullptr, r0, nrows);
}
// Second: x2 and one of query, key, value per workgroup, grid (tiles, 3), or (tiles, 1) at the end of the chain; dynamic
// LDS: 16 rows of h.
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void layer_bridge_fwd_split2_kernel(const BridgeArgs P) {
    extern __shared__ __attribute__((aligned(16))) float s_dyn[];
    constexpr int D = 128 * CT, ldx = D + BR_PAD;
    using G = BridgeGroups<CT>;
    __shared__ __attribute__((aligned(16))) float s_x[16 * ldx];
    __shared__ __attribute__((aligned(16))) float s_x1[16 * ldx];
    __shared__ float s_turn[BR_WAVES * 16 * 17];
    const int lane = threadIdx.x & 63, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * 16, nrows = min(16, P.N - r0), part = blockIdx.y;
    const int chunks = P.F / BR_CHUNK, ldf = P.F + BR_PAD;
    const int g4 = G::HEAD + chunks * G::CHUNK + part * CT * CT;
    WeightStream ws;
    ws.start(P.stream, P.steps, G::HEAD + CT);
    bridge_rows<1>(P.h, P.F, r0, nrows, s_dyn);
    bridge_rows<1>(P.x1, D, r0, nrows, s_x1);
    v4f_b2 acc3[CT][1];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) bridge_zero(acc3[ct]);
    __syncthreads();
#pragma unroll 1
    for (int c0 = 0; c0 < chunks; c0++) {
        const int g = G::HEAD + c0 * G::CHUNK + CT;
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
            bridge_sum(ws, ct + 1 < CT ? g + ct + 1 : (c0 + 1 < chunks ? g + G::CHUNK : g4), s_dyn + col * ldf + 4 * kk + BR_CHUNK * c0, ldf,
                       acc3[ct]);
    }
    bridge_second_sum<1, CT>(P, acc3, s_x1, s_x, r0, nrows, part == 0);
    if (!P.qs) return;
    __syncthreads();
    bridge_inputs_stage<1, CT, false>(P, ws, g4, part * CT, (part + 1) * CT, s_x, s_turn, r0, nrows);
}

// The start of the chain: the atoms' embedding x0 = x We^T, x (N, feat), to x2, and the inputs of the first layer.  The
// rows of x, a few dozen columns and not 16-byte aligned, are staged word by word, zeros behind the last feature.
// grid (tiles of 16 rows, query / key / value or 1: all three); dynamic LDS: 16 (16 feature steps + BR_PAD) floats.
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void layer_front_fwd_kernel(const BridgeArgs P) {
    extern __shared__ __attribute__((aligned(16))) float s_dyn[];
    constexpr int TR = 1, D = 128 * CT, ldx = D + BR_PAD, R = 16;
    __shared__ __attribute__((aligned(16))) float s_x[R * ldx];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * R, nrows = min(R, P.N - r0);
    const int feat = P.feat, pad = 16 * bridge_feat_steps(feat), ldf = pad + BR_PAD, eg = pad / 128;
    const int parts = gridDim.y == 1 ? 3 : 1, part = blockIdx.y, g0 = CT * eg + part * CT * CT;
    WeightStream ws;
    ws.start(P.stream, P.steps, 0);
    for (int idx = threadIdx.x; idx < R * pad; idx += 64 * BR_WAVES) {
        const int m = idx / pad, c = idx - m * pad;
        s_dyn[m * ldf + c] = m < nrows && c < feat ? P.attn[(size_t)(r0 + m) * feat + c] : 0.0f;
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
            bridge_sum(ws, at + 1 < CT * eg ? at + 1 : g0, s_dyn + col * ldf + 4 * kk + 128 * g, ldf, acc);
        }
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                s_x[m * ldx + n] = acc[tr][c];
                if (part == 0 && m < nrows) P.x2[(size_t)(r0 + m) * D + n] = acc[tr][c];
            }
    }
    __syncthreads();
    bridge_inputs_stage<TR, CT, true>(P, ws, g0, part * CT, (part + parts) * CT, s_x, nullptr, r0, nrows);
}

// ---- backward ------------------------------------------------------------------------------------------------
struct BridgeBwdArgs {
    const float* g_x2;            // (N, D) or null (zero)
    const float* gqkv;            // (N, 3 D), or null: made from ai_* below, or (those null as well) no next layer: g2 = g_x2
    const float* h;               // (N, F) forward activations (the rectifier's mask)
    const float* stream; int steps;
    float* g2; float* gh; float* g1; float* g_attn;                         // (N, D), (N, F), (N, D), (N, D)
    int N, F, H;
    int inputs_only;              // the first layer: g2 = g_x2 + gqkv Wqkv and no more
    int klen_q, klen_h, klen_1, klen_o;      // slices of the four sums over k
    // optional: the backward of attention_inputs.hpp for the rows of the workgroup, its result written to gqkv_out for the
    // weight-gradient launch
    const float* ai_qkv;          // (N, 3 D) forward projection output
    const float* ai_w; const float* ai_gauss;
    const float* ai_gqs; const float* ai_gk; const float* ai_gv; const float* ai_ga;    // each may be null (zero)
    float* gqkv_out;              // (N, 3 D)
    float* gw_partial;            // (ceil(N / 16), D): per 16 rows the sum of the lattice-weight gradient
    float c1, lb, c2, q_scale;
};
// The rows of gqkv into s_q (LDS), read or made from the gradients of the attention inputs (s_qf: LDS [R][D + BR_PAD],
// s_ga: LDS [R][H]); with `store` also to memory, with the partial sums of the lattice-weight gradient.
template <int TR, int CT>
__device__ __forceinline__ void bridge_bwd_inputs(const BridgeBwdArgs& P, float* s_q, float* s_qf, float* s_ga, int r0, int nrows,
                                                  bool store) {
    constexpr int D = 128 * CT, Q = 3 * D, ldx = D + BR_PAD, ldq = Q + BR_PAD, R = 16 * TR;
    if (!P.ai_qkv) {
        bridge_rows<TR>(P.gqkv, Q, r0, nrows, s_q);
        return;
    }
    for (int idx = threadIdx.x * 4; idx < R * D; idx += 64 * BR_WAVES * 4) {
        const int m = idx / D, c = idx - m * D;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < nrows) v = *reinterpret_cast<const float4*>(P.ai_qkv + (size_t)(r0 + m) * Q + c);
        *reinterpret_cast<float4*>(s_qf + m * ldx + c) = v;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < R * P.H; t += 64 * BR_WAVES) {
        const int m = t / P.H, hh = t - m * P.H;
        float galpha = 0.0f;
        if (m < nrows && P.ai_ga) {
            float alpha = 0.0f, scale = 1.0f;
#pragma unroll
            for (int d = 0; d < DH; d++) alpha = fmaf(s_qf[m * ldx + hh * DH + d], P.ai_w[hh * DH + d], alpha);
            if (P.ai_gauss) { scale = P.ai_gauss[0]; alpha = (alpha + P.ai_gauss[1]) * scale; }
            const float u = alpha * P.c1;
            const float e = u > 0.0f ? u : expm1f(u);
            const float slope = (u > 0.0f ? 1.0f : e + 1.0f) * P.c1 * scale * (1.0f - P.lb) * P.c2;
            galpha = P.ai_ga[(size_t)(r0 + m) * P.H + hh] * slope;
        }
        s_ga[m * P.H + hh] = galpha;
    }
    __syncthreads();
    for (int idx = threadIdx.x * 4; idx < R * Q; idx += 64 * BR_WAVES * 4) {
        const int m = idx / Q, c = idx - m * Q;
        const int which = c / D, cc = c - which * D;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < nrows) {
            const float* up = which == 0 ? P.ai_gqs : (which == 1 ? P.ai_gk : P.ai_gv);
            if (up) v = *reinterpret_cast<const float4*>(up + (size_t)(r0 + m) * D + cc);
            if (which == 0) {
                const float ga = s_ga[m * P.H + (cc >> 4)];
                const float4 w4 = *reinterpret_cast<const float4*>(P.ai_w + cc);
                v.x = fmaf(ga, w4.x, v.x * P.q_scale); v.y = fmaf(ga, w4.y, v.y * P.q_scale);
                v.z = fmaf(ga, w4.z, v.z * P.q_scale); v.w = fmaf(ga, w4.w, v.w * P.q_scale);
            }
            if (store) *reinterpret_cast<float4*>(P.gqkv_out + (size_t)(r0 + m) * Q + c) = v;
        }
        *reinterpret_cast<float4*>(s_q + m * ldq + c) = v;
    }
    if (store)
        for (int t = threadIdx.x; t < TR * D; t += 64 * BR_WAVES) {
            const int tr = t / D, c = t - tr * D;
            if (16 * tr >= nrows) continue;
            float part = 0.0f;
#pragma unroll
            for (int m = 0; m < 16; m++) part = fmaf(s_ga[(16 * tr + m) * P.H + (c >> 4)], s_qf[(16 * tr + m) * ldx + c], part);
            P.gw_partial[(size_t)(blockIdx.x * TR + tr) * D + c] = part;
        }
}
// g2 = g_x2 + gqkv Wqkv into s_g2 and, with `store`, memory.  `then`: the group behind the stage's 3 CT^2.
template <int TR, int CT>
__device__ __forceinline__ void bridge_bwd_first(const BridgeBwdArgs& P, WeightStream& ws, int then, const float* s_q, float* s_g2, int r0,
                                                 int nrows, bool store) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD, ldq = 3 * D + BR_PAD;
#pragma unroll 1
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        float add[TR][4];
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                add[tr][c] = P.g_x2 && m < nrows ? P.g_x2[(size_t)(r0 + m) * D + n] : 0.0f;
            }
        v4f_b2 acc[TR], sum[TR];
        bridge_zero(acc);
        int in_slice = 0;
        bool first = true;
#pragma unroll 1
        for (int g = 0; g < 3 * CT; g++) {
            const int at = ct * 3 * CT + g;
            bridge_steps<TR, true>(ws, at + 1 < 3 * CT * CT ? at + 1 : then, s_q + col * ldq + 4 * kk + 128 * g, ldq, acc, sum, P.klen_q,
                                   in_slice, first);
        }
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                float val = sum[tr][c];
                if (P.g_x2) val += add[tr][c];
                s_g2[m * ldx + n] = val;
                if (store && m < nrows) P.g2[(size_t)(r0 + m) * D + n] = val;
            }
    }
}
// Chunk c0 of gh (its groups start at g) from s_g2, into hb (LDS) if given and to memory.
template <int TR, int CT>
__device__ __forceinline__ void bridge_bwd_chunk(const BridgeBwdArgs& P, WeightStream& ws, int c0, int g, int then, const float* s_g2,
                                                 float* hb, int r0, int nrows) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD, ldh = BR_CHUNK + BR_PAD;
    const int n = BR_CHUNK * c0 + 16 * wave + col;
    float mask[TR][4];
#pragma unroll
    for (int tr = 0; tr < TR; tr++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int m = 16 * tr + 4 * kk + c;
            mask[tr][c] = m < nrows ? P.h[(size_t)(r0 + m) * P.F + n] : 0.0f;
        }
    v4f_b2 acc[TR], sum[TR];
    bridge_zero(acc);
    int in_slice = 0;
    bool first = true;
#pragma unroll
    for (int i = 0; i < CT; i++)
        bridge_steps<TR, true>(ws, i + 1 < CT ? g + i + 1 : then, s_g2 + col * ldx + 4 * kk + 128 * i, ldx, acc, sum, P.klen_h, in_slice,
                               first);
#pragma unroll
    for (int tr = 0; tr < TR; tr++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int m = 16 * tr + 4 * kk + c;
            const float val = mask[tr][c] > 0.0f ? sum[tr][c] : 0.0f;
            if (hb) hb[m * ldh + 16 * wave + col] = val;
            if (m < nrows) P.gh[(size_t)(r0 + m) * P.F + n] = val;
        }
}
template <int TR, int CT>
struct BridgeSliced {             // sums over the whole of F, in slices, chunk by chunk
    v4f_b2 acc[CT][TR], sum[CT][TR];
    int in_slice[CT];
    bool first[CT];
    __device__ __forceinline__ void start() {
#pragma unroll
        for (int ct = 0; ct < CT; ct++) { bridge_zero(acc[ct]); in_slice[ct] = 0; first[ct] = true; }
    }
};
// g1 = sums + g2 (s_g2) into s_g1 and memory, then g_attn = g1 Wo; the groups of Wo start at g.
template <int TR, int CT>
__device__ __forceinline__ void bridge_bwd_last(const BridgeBwdArgs& P, WeightStream& ws, int g, BridgeSliced<TR, CT>& S, const float* s_g2,
                                                float* s_g1, int r0, int nrows) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    constexpr int D = 128 * CT, ldx = D + BR_PAD;
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                const float val = S.sum[ct][tr][c] + s_g2[m * ldx + n];
                s_g1[m * ldx + n] = val;
                if (m < nrows) P.g1[(size_t)(r0 + m) * D + n] = val;
            }
    }
    __syncthreads();
#pragma unroll 1
    for (int ct = 0; ct < CT; ct++) {
        const int n = 16 * (8 * ct + wave) + col;
        v4f_b2 acc[TR], sum[TR];
        bridge_zero(acc);
        int in_slice = 0;
        bool first = true;
#pragma unroll
        for (int i = 0; i < CT; i++)
            bridge_steps<TR, true>(ws, ++g, s_g1 + col * ldx + 4 * kk + 128 * i, ldx, acc, sum, P.klen_o, in_slice, first);
#pragma unroll
        for (int tr = 0; tr < TR; tr++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const int m = 16 * tr + 4 * kk + c;
                if (m < nrows) P.g_attn[(size_t)(r0 + m) * D + n] = sum[tr][c];
            }
    }
}

// grid: ceil(N / (16 TR)) workgroups of 512 threads.  128 registers (CT = 1), so that a compute unit holds two workgroups:
// 155 us at 22 528 rows with the 130 that the compiler takes by itself, 128 us with 128.
template <int TR, int CT>
__global__ __launch_bounds__(64 * BR_WAVES, 4 / CT) void layer_bridge_bwd_kernel(const BridgeBwdArgs P) {
    constexpr int D = 128 * CT, ldx = D + BR_PAD, ldq = 3 * D + BR_PAD, ldh = BR_CHUNK + BR_PAD, R = 16 * TR;
    __shared__ __attribute__((aligned(16))) float s_q[R * ldq];           // gqkv; later the chunks of gh
    __shared__ __attribute__((aligned(16))) float s_g2[R * ldx];
    __shared__ __attribute__((aligned(16))) float s_g1[R * ldx];          // (the forward query rows at first)
    __shared__ float s_ga[R * 8 * CT];
    static_assert(ldq >= 2 * ldh, "two chunks of gh fit the place of gqkv");
    const int lane = threadIdx.x & 63, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * R, nrows = min(R, P.N - r0);
    const bool next = P.gqkv != nullptr || P.ai_qkv != nullptr;
    const int head = next ? 3 * CT * CT : 0, chunks = P.F / BR_CHUNK;
    WeightStream ws;
    ws.start(P.stream, P.steps, 0);
    if (next) {
        bridge_bwd_inputs<TR, CT>(P, s_q, s_g1, s_ga, r0, nrows, true);
        __syncthreads();
        bridge_bwd_first<TR, CT>(P, ws, head, s_q, s_g2, r0, nrows, true);
        if (P.inputs_only) return;
    } else if (P.g_x2) {
        bridge_rows<TR>(P.g_x2, D, r0, nrows, s_g2);
    } else {
        for (int idx = threadIdx.x; idx < R * ldx; idx += 64 * BR_WAVES) s_g2[idx] = 0.0f;
    }
    __syncthreads();
    BridgeSliced<TR, CT> S;
    S.start();
#pragma unroll 1
    for (int c0 = 0; c0 < chunks; c0++) {
        float* const hb = s_q + (c0 & 1) * (R * ldh);
        const int g = head + c0 * 2 * CT;
        bridge_bwd_chunk<TR, CT>(P, ws, c0, g, g + CT, s_g2, hb, r0, nrows);
        __syncthreads();          // (the other chunk buffer was last read before the barrier of the chunk in between)
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
            bridge_steps<TR, true>(ws, g + CT + ct + 1, hb + col * ldh + 4 * kk, ldh, S.acc[ct], S.sum[ct], P.klen_1, S.in_slice[ct],
                                   S.first[ct]);
    }
    bridge_bwd_last<TR, CT>(P, ws, head + chunks * 2 * CT, S, s_g2, s_g1, r0, nrows);
}
// The same chain in two launches, for few rows.  First: g2 and one chunk of gh per workgroup, grid (tiles of 16 rows, chunks).
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void layer_bridge_bwd_split1_kernel(const BridgeBwdArgs P) {
    constexpr int D = 128 * CT, ldx = D + BR_PAD, ldq = 3 * D + BR_PAD;
    __shared__ __attribute__((aligned(16))) float s_q[16 * ldq];
    __shared__ __attribute__((aligned(16))) float s_g2[16 * ldx];
    __shared__ __attribute__((aligned(16))) float s_qf[16 * ldx];
    __shared__ float s_ga[16 * 8 * CT];
    const int r0 = blockIdx.x * 16, nrows = min(16, P.N - r0), c0 = blockIdx.y;
    const bool next = P.gqkv != nullptr || P.ai_qkv != nullptr;
    const int head = next ? 3 * CT * CT : 0, g = head + c0 * 2 * CT;
    WeightStream ws;
    ws.start(P.stream, P.steps, next ? 0 : g);
    if (next) {
        bridge_bwd_inputs<1, CT>(P, s_q, s_qf, s_ga, r0, nrows, c0 == 0);
        __syncthreads();
        bridge_bwd_first<1, CT>(P, ws, g, s_q, s_g2, r0, nrows, c0 == 0);
    } else if (P.g_x2) {
        bridge_rows<1>(P.g_x2, D, r0, nrows, s_g2);
    } else {
        for (int idx = threadIdx.x; idx < 16 * ldx; idx += 64 * BR_WAVES) s_g2[idx] = 0.0f;
    }
    __syncthreads();
    bridge_bwd_chunk<1, CT>(P, ws, c0, g, g, s_g2, nullptr, r0, nrows);
}
// Second: g1 and g_attn, grid (tiles); dynamic LDS: 16 rows of gh.
template <int CT>
__global__ __launch_bounds__(64 * BR_WAVES) void layer_bridge_bwd_split2_kernel(const BridgeBwdArgs P) {
    extern __shared__ __attribute__((aligned(16))) float s_dyn[];
    constexpr int D = 128 * CT, ldx = D + BR_PAD;
    __shared__ __attribute__((aligned(16))) float s_g2[16 * ldx];
    __shared__ __attribute__((aligned(16))) float s_g1[16 * ldx];
    const int lane = threadIdx.x & 63, col = lane & 15, kk = lane >> 4;
    const int r0 = blockIdx.x * 16, nrows = min(16, P.N - r0);
    const bool next = P.gqkv != nullptr || P.ai_qkv != nullptr;
    const int head = next ? 3 * CT * CT : 0, chunks = P.F / BR_CHUNK, ldf = P.F + BR_PAD;
    WeightStream ws;
    ws.start(P.stream, P.steps, head + CT);
    bridge_rows<1>(P.gh, P.F, r0, nrows, s_dyn);
    const float* const g2 = next ? P.g2 : P.g_x2;
    if (g2) bridge_rows<1>(g2, D, r0, nrows, s_g2);
    else
        for (int idx = threadIdx.x; idx < 16 * ldx; idx += 64 * BR_WAVES) s_g2[idx] = 0.0f;
    __syncthreads();
    BridgeSliced<1, CT> S;
    S.start();
    const int g4 = head + chunks * 2 * CT;
#pragma unroll 1
    for (int c0 = 0; c0 < chunks; c0++) {
        const int g = head + c0 * 2 * CT + CT;
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
            bridge_steps<1, true>(ws, ct + 1 < CT ? g + ct + 1 : (c0 + 1 < chunks ? g + 2 * CT : g4),
                                  s_dyn + col * ldf + 4 * kk + BR_CHUNK * c0, ldf, S.acc[ct], S.sum[ct], P.klen_1, S.in_slice[ct],
                                  S.first[ct]);
    }
    bridge_bwd_last<1, CT>(P, ws, g4, S, s_g2, s_g1, r0, nrows);
}

}  // namespace cfh
