// Fused attention core: lattice sums, softmax over the pairs of an atom and the value encoding in ONE pass per
// (atom i, head h), with ONE histogram per (atom, head) instead of one per (pair, head).
//
// The attention output is linear in the value encoding,
//     out_i = sum_j P_ij (v_j + psi_ij),   psi_ij = W . shat_ij,   shat_ij = sum_n p_n b(image n of pair ij),
// so  sum_j P_ij psi_ij = W . T_i  with  T_i = sum_j sum_n P_ij p_n b(.): the per-image basis values can be
// scattered, weighted by P_ij p_n, into one histogram per item, and the projection W is applied once per item by
// a small MFMA product afterwards.  psi (E,H,16) and the per-pair histograms never exist.  The softmax weights
// P_ij are not known before all pairs of the row have been seen, so the pass keeps a running maximum of the
// logits (q_i.k_j + z_ij) and rescales histogram, value accumulator and denominator when it grows (online
// softmax).  What the reference computes in five kernels and a tensor sum
// (models/kernels/real_enc_frame_proj_fwd_length.cu, ..._fwd_angle.cu, fused_dpa_fwd.cu;
//  models/cuda_funcs/real_space_framed_proj.py:21-120, fused_dpa.py:17-63) is one kernel plus the projection here.
//
// Two further changes of formulation (same mathematics, different arithmetic):
//   * sorted translations.  For the usual box (half-width 2 = 125 translations) a table of the box's shifts
//     sorted by length is made once per crystal.  An image at shift s of a pair at r lies at distance
//     >= |s| - |r|, so the nearest image of a pair is found in the prefix |s| <= 2|r| and every image whose
//     weight can reach 2^-skip of the heaviest one in the prefix |s| <= |r| + sqrt(d2min + skip/(-a log2 e)):
//     the two light sweeps read a fraction of the box instead of all of it twice.
//   * angle encoding by local moments.  The Gaussian basis of the cosine has sigma = wscale bins (4), so around
//     the bin m* nearest to x the value of every basis function is a short power series in the offset
//     eps = 2 (u - m*) in [-1,1] (u = x in bin units):
//         exp(-((m - u)/ws)^2 / 2) = sum_o eps^o D_o(m - m*),  D_o(d) = exp(-(d/ws)^2/2) He_o(d/ws) / (o! (2 ws)^o)
//     (generating function of the Hermite polynomials; truncated after NORD = 5 terms the error is below 2e-6 of
//     the peak, 6 terms: 1e-7).  A term therefore adds NORD moments w eps^o at ONE bin per axis instead of a 33-bin window, and
//     the constant matrices D_o are folded into the projection weights (core_wcat_kernel).  This is the FULL
//     basis (no +-4 sigma truncation), i.e. the pure-PyTorch formulation of the reference
//     (models/indexed_lattice_multi_head_attention.py:580-588) rather than the windowed one of its CUDA kernels.
//     The distance basis (sigma = 1 bin) keeps its truncated window.
//
// Histogram of an item ("hist", HW words): [0,64) distance bins, then for axis ax and order o the 64 moment bins
// at 64 + (ax NORD + o) 64.  It is accumulated in LDS as signed 32-bit fixed point (round to nearest) in units of
// 2^30 / npairs relative to the heaviest pair of the row so far, and written out normalised as float32.
#pragma once
#include <type_traits>
#include "device_common.hpp"
#include "moment_series.hpp"

namespace cfh {

constexpr int FC_TCAP = 128;                    // translations per table chunk (the sorted table of the usual box fits)
constexpr int FC_GROUP = 8;                     // pairs per group: one per 8-lane row
constexpr int FC_LISTCAP = FC_GROUP * FC_TCAP;  // a group's survivors always fit: no overflow handling
constexpr int FC_SHIFT = 7;                     // list entry = pair-in-group << 7 | table index
constexpr int FC_BIGSHIFT = 13;                 // ... of an item of several chunks: pair-in-group << 13 | index in its box
constexpr int FC_BIGT = 1 << FC_BIGSHIFT;       // (boxes of up to 8192 translations)
constexpr int CORE_WPB = 1;                     // wavefronts per workgroup of the main kernels: each takes an item of its
                                                // own (no barriers).  Workgroups of 4 or 8 items of one head that make the
                                                // products with the head's weights themselves (projection, G) were slower:
                                                // +25 us per kernel for the phases behind barriers, against 21 + 20 us for
                                                // the two separate launches
constexpr int CORE_DIE_SHIFT = 3;               // frame search and main kernels: runs of 8 items, an atom's with 8 heads, on one die
                                                // (die_order): they share the pairs' geometry and the lines of k, v, z and P,
                                                // where item by item every die had a head.  Whole passes: training step of
                                                // 18 976 items 1279 -> 1265 us, with 16 angle bins 1260 -> 1237, cells of 40 to
                                                // 200 atoms 1146 -> 1132, inference of 180 224 items 3033 -> 3026
constexpr int FC_LOGCAP = 64;                   // logits of a row kept in LDS until the row is complete
constexpr int HW_DIST = NBINS;
constexpr int HW_ANG = NBINS * (1 + 3 * NORD);  // 1024 words per (atom, head) with the 64-bin angle encoding
constexpr int SMALL_A = 16;                     // the 16-bin angle basis (the reference's lightweight setting): sigma is
                                                // one bin or more, far too wide a step for the moment series, and the
                                                // basis is small: every image adds its 16 basis values per axis directly
                                                // (the whole basis, as the reference evaluates it for 16 bins)
constexpr int HW_ANG16 = 2 * NBINS;             // 64 distance bins + 3 axes x 16 bins, padded to whole 64-word blocks
// In LDS the 3 x 16 angle bins of an item exist A16_COPIES times, one copy per value of lane & 15: every image adds
// to ALL 16 bins of an axis in the same order, so with one copy the 64 lanes of an atomic instruction would meet on
// one word (128 clocks instead of 6).  A copy has an odd number of words so that the copies start in different banks.
constexpr int A16_COPIES = 16;
constexpr int A16_STRIDE = 3 * SMALL_A + 1;
// words of an item's histogram in LDS
__host__ __device__ constexpr int core_hist_lds_words(int ang) {
    return ang == SMALL_A ? HW_DIST + A16_COPIES * A16_STRIDE : (ang == NBINS ? HW_ANG : HW_DIST);
}
// words of an item's histogram for `ang` angle bins (0: distance encoding alone)
__host__ __device__ constexpr int core_hist_words(int ang, bool lean = false);
// Inference, where the histogram serves the projection alone, uses FEWER nodes for the moments of the angle encoding than
// one per bin (moment_series.hpp): 720 words instead of 1024, with an error of the series that is no larger.  At 22 528 atoms:
// projection 204 -> 131 us, main kernel 404 -> 383 (its vector instructions, not its stores, bound it; making the projection
// in it, four items of a head per workgroup behind a barrier, took 529 us for both at 640 words).
constexpr int HW_LEAN = 720;
static_assert(HW_LEAN >= HW_DIST + 3 * NORD * LEAN_NODES && HW_LEAN % 16 == 0, "");
__host__ __device__ constexpr int core_hist_words(int ang, bool lean) {
    return ang == NBINS ? (lean ? HW_LEAN : HW_ANG) : (ang == SMALL_A ? HW_ANG16 : HW_DIST);
}
constexpr int REC_J0 = 30;                      // item record: first neighbour atom (pairs of an atom are j0, j0+1, ...)
constexpr int REC_CRYSTAL = 31;                 // item record: crystal of the atom
static_assert(FC_TCAP == (1 << FC_SHIFT) && (FC_GROUP << FC_SHIFT) <= 65536, "list entry is 16 bits");

typedef float v4f_c __attribute__((ext_vector_type(4)));

// Optional phase timing (compile with -DCFH_PHASE_TIMING; diagnostics builds only): cycles per phase of the forward
// kernel, summed over the wavefronts, in the statistics slots 16..23.
#ifdef CFH_PHASE_TIMING
#define CFH_PH_DECL unsigned long long ph_acc[8] = {0, 0, 0, 0, 0, 0, 0, 0}; unsigned long long ph_last = __builtin_amdgcn_s_memtime(); int ph_cur = 0;
#define CFH_PH(n) do { const unsigned long long ph_t = __builtin_amdgcn_s_memtime(); ph_acc[ph_cur] += ph_t - ph_last; ph_last = ph_t; ph_cur = (n); } while (0)
#define CFH_PH_FLUSH(stats) do { CFH_PH(0); if ((stats) && (threadIdx.x & 63) == 0) for (int u = 0; u < 8; u++) atomicAdd((stats) + 16 + u, ph_acc[u]); } while (0)
#else
#define CFH_PH_DECL
#define CFH_PH(n) do { } while (0)
#define CFH_PH_FLUSH(stats) do { } while (0)
#endif

struct CoreArgs {
    KernelArgs K;                 // geometry, work queues, item records, basis constants
    const float* qs;              // (N,H,16) query, already divided by sqrt(16)
    const float* k;               // (N,H,16)
    const float* v;               // (N,H,16)
    const float4* sorted_tab;     // (B, FC_TCAP) shifts of the usual box sorted by length, w = length; or null
    const float2* pair_near;      // (E) per pair over that box: smallest d^2 of all images, of the images with
                                  // d^2 > 1e-5 (what the frame search may point at; low 7 bits: that image's
                                  // position in the sorted table); or null
    int32_t table_R;              // half-width that table was made for
    int32_t slow_wgs;             // leading wavefronts of the main kernels that take the listed slow records first, by
                                  // rank over all lists: wavefront w the rank w; the listed records of higher rank are
                                  // taken in place, like the others (0: no lists)
    int32_t slow_lists;           // lists (K.slow_count, K.slow_list)
    int32_t slow_stride;          // slots per list
    uint32_t slow_flag;           // the flag in the box word of the records listed for this launch
    float skip_log2;              // images lighter than 2^-skip of the heaviest of their pair are not visited (<= 0: all are)
    // forward results
    float* out;                   // (N,H,16) sum_j P_ij v_j (core_project_kernel adds W . hist)
    float* prob;                  // (E,H) P_ij
    float* z;                     // (E,H)
    float* hist;                  // (H,N,hw); inference with angles: (H, 16 sixteens(N), hw), row 16 sixteen_of(it) + rank
    const float* wcat;            // (H,16,hw) weights of the products (with `tickets`)
    int32_t* tickets;             // per (16 items, head) how many of them are done (core_project_done); or null
    int32_t ticket_items;         // the places of the work order, from the start, that draw tickets
    // backward operands and results
    const float* go;              // (N,H,16) upstream gradient of out
    const float* outv;            // (N,H,16) the forward's final out
    const float* G;               // (H,N,hw) Wcat^T go per item
    float* gq;                    // (N,H,16)
    float* glogit;                // (E,H) gradient of the logits (the column kernel turns it into gk)
};

// Loads at a 32-bit BYTE offset from a base that is the same in all lanes: the address is (scalar base + vector offset),
// one instruction's operands, where an element index of 64 bits costs two or three vector instructions per address
// (the entry points refuse sizes whose offsets would not fit).
template <typename T>
__device__ __forceinline__ T load_at(const void* base, uint32_t byte_off) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}

// ---- reductions over an 8-lane row (half of a DPP row) -------------------------------------------------------
__device__ __forceinline__ float half_sum(float x) {
    x += dpp_move<0xB1>(x); x += dpp_move<0x4E>(x); x += dpp_move<0x141>(x); return x;
}
__device__ __forceinline__ float half_min(float x) {
    x = fminf(x, dpp_move<0xB1>(x)); x = fminf(x, dpp_move<0x4E>(x)); x = fminf(x, dpp_move<0x141>(x)); return x;
}
__device__ __forceinline__ float wave_maxf(float v) { return -wave_min(-v); }
// sum over the 8 rows for every position in the row: lanes s, s+8, ..., s+56
__device__ __forceinline__ float rows8_sum(float x) {
    x += dpp_move<0x128>(x);          // row_ror 8: the other half of the 16-lane row
    return rows_sum(x);
}
// float -> fixed point, round to nearest (floor(x + 0.5)) in ONE instruction (rintf + conversion are two)
__device__ __forceinline__ int rint_i(float x) {
    int r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// ---- sorted shifts of the usual box, one table per crystal ---------------------------------------------------
// block = crystal, 128 threads; entry = (shift, |shift|), ascending length (ties: loop order); entries beyond the
// box: length +inf.  The low 7 bits of the length hold the translation's index in the reference's loop order (the
// frame search breaks ties by it): the length is rounded down by at most 2^-16 of itself, which the margins of every
// reach test cover.
__device__ __forceinline__ void sorted_shifts_block(const float* __restrict__ tvecs, int R0, float4* __restrict__ out, int b, int t,
                                                    float* key) {
    const int s = 2 * R0 + 1, T0 = s * s * s;
    float4 v = make_float4(0.f, 0.f, 0.f, __builtin_inff());
    if (t < T0) {
        const float* L = tvecs + (size_t)b * 9;
        const float n3 = (float)(t % s - R0), n2 = (float)((t / s) % s - R0), n1 = (float)(t / (s * s) - R0);
        v.x = fmaf(L[6], n3, fmaf(L[3], n2, L[0] * n1));
        v.y = fmaf(L[7], n3, fmaf(L[4], n2, L[1] * n1));
        v.z = fmaf(L[8], n3, fmaf(L[5], n2, L[2] * n1));
        v.w = sqrtf(fmaf(v.x, v.x, fmaf(v.y, v.y, v.z * v.z)));
    }
    key[t] = v.w;
    __syncthreads();
    int rank = 0;
    for (int u = 0; u < FC_TCAP; u++) {
        const float ku = key[u];
        rank += (ku < v.w || (ku == v.w && u < t)) ? 1 : 0;
    }
    if (t < T0) v.w = __uint_as_float((__float_as_uint(v.w) & ~(uint32_t)(FC_TCAP - 1)) | (uint32_t)t);
    out[(size_t)b * FC_TCAP + rank] = v;
}
__global__ __launch_bounds__(FC_TCAP) void sorted_shifts_kernel(const float* __restrict__ tvecs, int R0, float4* __restrict__ out) {
    __shared__ float key[FC_TCAP];
    sorted_shifts_block(tvecs, R0, out, (int)blockIdx.x, (int)threadIdx.x, key);
}

// Per pair, over the usual box of its crystal: the smallest squared distance of all images and of the images with
// d^2 > 1e-5, the latter with the position of that image in the sorted table in its low 7 bits.  Both depend on the geometry alone, not on the head or the layer, so they are made once per batch:
// the lattice sums of an item with the usual box then need no sweep for the nearest image, and the frame search
// knows how far into the sorted table a pair's best first-axis candidate can sit.  Eight lanes per pair, eight
// entries of the sorted table at a time; the sorted order ends the loop once |s| - |r| exceeds the larger of the
// two minima (an entry behind that point cannot lower either minimum, so taking the rest of its group of eight
// along changes nothing).  Same arithmetic for d^2 as the sweeps.  A thread per pair walking the table alone took
// 16 us for its chain of dependent steps; this takes 7.
__device__ __forceinline__ float2 pair_nearest(float rx, float ry, float rz, const float4* tab, int T0, int sub) {
    const float r = hw_sqrt(fmaf(rx, rx, fmaf(ry, ry, rz * rz)));      // (here and below a bound with margins)
    // (dval carries the table position of its image in its low 7 bits -- it is rounded down by at most 2^-16 of itself,
    // which the margins of every test that uses it cover -- so that the minimum over the lanes brings the position along)
    float dall = 3.0e38f, dval = 3.0e38f;
    float4 v = tab[sub];
    float w = tab[0].w;
    for (int t0 = 0; t0 < T0; t0 += 8) {
        // the first entry of the group decides for all eight lanes whether the walk goes on
        if (dval < 1.0e38f && w > fmaf(1.0001f, r + hw_sqrt(dval), 1e-3f)) break;
        const int next = min(t0 + 8, FC_TCAP - 8);           // (the next group's entries, in flight meanwhile)
        const float4 vn = tab[next + sub];
        const float wn = tab[next].w;
        if (t0 + sub < T0) {
            const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
            const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            dall = fminf(dall, d2);
            if (d2 > 1e-5f)
                dval = fminf(dval, __uint_as_float((__float_as_uint(d2) & ~(uint32_t)(FC_TCAP - 1)) | (uint32_t)(t0 + sub)));
        }
        dall = half_min(dall);
        dval = half_min(dval);
        v = vn; w = wn;
    }
    return make_float2(dall, dval);
}
__global__ __launch_bounds__(256) void pair_nearest_kernel(const float* __restrict__ rpos, const int64_t* __restrict__ edges,
                                                           const int64_t* __restrict__ batch,
                                                           const float4* __restrict__ sorted_tab, int T0, int E,
                                                           float2* __restrict__ out) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int e = min(g >> 3, E - 1), sub = g & 7;       // (the lanes of a group past the end redo the last pair)
    const float2 near = pair_nearest(rpos[(size_t)e * 3 + 0], rpos[(size_t)e * 3 + 1], rpos[(size_t)e * 3 + 2],
                                     sorted_tab + (size_t)batch[edges[e]] * FC_TCAP, T0, sub);
    if (sub == 0 && (g >> 3) < E) out[e] = near;
}

// ---- projection weights with the moment matrices folded in ---------------------------------------------------
// table of D_o(d) for d = -63 .. 63 in LDS, made by the threads of a block: dtab[o * 128 + d + 63]
__device__ __forceinline__ void build_moment_table(float* dtab, float ws) {
    for (int u = threadIdx.x; u < NORD * 128; u += blockDim.x) {
        const int o = u >> 7, d = (u & 127) - 63;
        dtab[u] = (u & 127) < 127 ? moment_matrix<float>(o, (float)d, ws) : 0.0f;
    }
    __syncthreads();
}
// The same for the nodes of inference: dtab[o * LEAN_TAB + LEAN_DEN m - LEAN_NUM n + LEAN_OFF] = coefficient of eps^o
// around node n of the basis function of bin m.
constexpr int LEAN_OFF = LEAN_NUM * (LEAN_NODES - 1), LEAN_TAB = LEAN_OFF + LEAN_DEN * NBINS;
__device__ __forceinline__ void build_node_table(float* dtab, float ws) {
    const float r = 0.5f * LEAN_NUM / LEAN_DEN / ws, inv_ws = 1.0f / ws;
    for (int u = threadIdx.x; u < LEAN_TAB; u += blockDim.x) {
        float c[NORD];
        node_coefficients((float)(u - LEAN_OFF) * (1.0f / LEAN_DEN) * inv_ws, r, c);
#pragma unroll
        for (int o = 0; o < NORD; o++) dtab[o * LEAN_TAB + u] = c[o];
    }
    __syncthreads();
}
// wcat (H,16,hw): [0,64) dist_coef W_dist;  64 + (ax NORD + o) 64 + m': angle_coef sum_m W_ax[c,m] D_o(m - m').
// grid: H*16 blocks (h, c), the threads over the words.
struct WcatArgs {
    const float* Wd; const float* W1; const float* W2; const float* W3;      // (H,16,64) and (H,16,A) x 3
    int hw;
    float dist_coef, angle_coef, ws;
    float* wcat;
};
__device__ __forceinline__ void core_wcat_block(const WcatArgs& A, int hc) {
    const float* __restrict__ Wd = A.Wd; const float* __restrict__ W1 = A.W1;
    const float* __restrict__ W2 = A.W2; const float* __restrict__ W3 = A.W3;
    const int hw = A.hw;
    const float dist_coef = A.dist_coef, angle_coef = A.angle_coef, ws = A.ws;
    float* __restrict__ wcat = A.wcat;
    __shared__ float row[3][NBINS];
    __shared__ float dtab[NORD * LEAN_TAB];
    if (hw == HW_ANG16) {
        // 16-bin basis: the weights themselves behind the distance block, zeros in the padding
        for (int w = threadIdx.x; w < hw; w += blockDim.x) {
            float val = 0.0f;
            if (w < HW_DIST) val = dist_coef * Wd[(size_t)hc * NBINS + w];
            else if (w < HW_DIST + 3 * SMALL_A) {
                const int u = w - HW_DIST, ax = u / SMALL_A, m = u % SMALL_A;
                const float* W = ax == 0 ? W1 : (ax == 1 ? W2 : W3);
                val = angle_coef * W[(size_t)hc * SMALL_A + m];
            }
            wcat[(size_t)hc * hw + w] = val;
        }
        return;
    }
    if (hw > HW_DIST) {
        for (int u = threadIdx.x; u < 3 * NBINS; u += blockDim.x) {
            const float* W = u < NBINS ? W1 : (u < 2 * NBINS ? W2 : W3);
            row[u / NBINS][u % NBINS] = W[(size_t)hc * NBINS + (u % NBINS)];
        }
        if (hw == HW_LEAN) build_node_table(dtab, ws);
        else build_moment_table(dtab, ws);
    }
    for (int w = threadIdx.x; w < hw; w += blockDim.x) {
        float val;
        if (w < HW_DIST) val = dist_coef * Wd[(size_t)hc * NBINS + w];
        else if (hw == HW_LEAN) {
            const int u = w - HW_DIST, ax = u / (NORD * LEAN_NODES), o = (u / LEAN_NODES) % NORD, n = u % LEAN_NODES;
            const float* dt = dtab + o * LEAN_TAB + LEAN_OFF - LEAN_NUM * n;
            float acc = 0.0f;
            if (ax < 3) {                  // (words past the last node: zero)
#pragma unroll 8
                for (int m = 0; m < NBINS; m++) acc = fmaf(row[ax][m], dt[LEAN_DEN * m], acc);
            }
            val = angle_coef * acc;
        } else {
            const int u = w - HW_DIST, ax = u / (NORD * NBINS), o = (u / NBINS) % NORD, mp = u % NBINS;
            const float* dt = dtab + o * 128 + 63 - mp;
            float acc = 0.0f;
#pragma unroll 8
            for (int m = 0; m < NBINS; m++) acc = fmaf(row[ax][m], dt[m], acc);
            val = angle_coef * acc;
        }
        wcat[(size_t)hc * hw + w] = val;
    }
}
__global__ __launch_bounds__(256) void core_wcat_kernel(const WcatArgs A) { core_wcat_block(A, (int)blockIdx.x); }
// The item records of a launch and the concatenated weights in ONE launch (neither depends on the other; both are a
// few microseconds of work behind a launch): the first prep_blocks workgroups are those of prepare_items_kernel, the
// following H * 16 those of core_wcat_kernel.
__global__ __launch_bounds__(256) void core_prepare_wcat_kernel(const KernelArgs P, int with_query, int prep_blocks,
                                                                const WcatArgs A) {
    if ((int)blockIdx.x < prep_blocks) prepare_items_block<true>(P, with_query, (int)blockIdx.x);
    else core_wcat_block(A, (int)blockIdx.x - prep_blocks);
}
constexpr int CORE_GW_SLICES = 8;      // at most this many slices of the atoms per job (copies of the scratch)
// A word's sum over the slices, in their order; all loads in flight at once.
__device__ __forceinline__ float core_slice_sum(const float* __restrict__ g, int nslices, size_t stride) {
    float v[CORE_GW_SLICES], sum = 0.0f;
#pragma unroll
    for (int sl = 0; sl < CORE_GW_SLICES; sl++) v[sl] = g[min(sl, nslices - 1) * stride];
#pragma unroll
    for (int sl = 0; sl < CORE_GW_SLICES; sl++) sum += sl < nslices ? v[sl] : 0.0f;
    return sum;
}
// The way back: gW_dist = dist_coef gwcat[.., 0:64];  gW_ax[c,m] = angle_coef sum_{o,m'} gwcat[.., ax,o,m'] D_o(m - m').
// Block hc = (head, channel), 256 threads = (enc 0..3, bin m).  acc_dst: added to what the destinations hold.
__device__ __forceinline__ void core_gw_finish_block(const float* __restrict__ gwcat, int nslices, size_t slice_stride,
                                                     int hw, float dist_coef, float angle_coef, float ws,
                                                     float* __restrict__ gWd, float* __restrict__ gW1,
                                                     float* __restrict__ gW2, float* __restrict__ gW3, int hc, bool acc_dst) {
    __shared__ float dtab[NORD * 128];
    __shared__ float grow[3 * NORD * NBINS];
    const int enc = threadIdx.x >> 6, m = threadIdx.x & 63;
    const float* g = gwcat + (size_t)hc * hw;
    if (hw == HW_ANG16) {
        // 16-bin basis: thread (enc, m) sums the slices of its word; the axes' rows have 16 bins
        if (enc > 0 && m >= SMALL_A) return;
        float* dst = enc == 0 ? gWd : (enc == 1 ? gW1 : (enc == 2 ? gW2 : gW3));
        if (!dst) return;
        const int word = enc == 0 ? m : HW_DIST + (enc - 1) * SMALL_A + m;
        const float sum = core_slice_sum(g + word, nslices, slice_stride);
        float* d = dst + (size_t)hc * (enc == 0 ? NBINS : SMALL_A) + m;
        *d = (acc_dst ? *d : 0.0f) + (enc == 0 ? dist_coef : angle_coef) * sum;
        return;
    }
    if (hw > HW_DIST) {
        for (int u = threadIdx.x; u < 3 * NORD * NBINS; u += 256) {
            grow[u] = core_slice_sum(g + HW_DIST + u, nslices, slice_stride);
        }
        build_moment_table(dtab, ws);
    }
    if (enc == 0) {
        if (gWd) {
            const float sum = core_slice_sum(g + m, nslices, slice_stride);
            float* d = gWd + (size_t)hc * NBINS + m;
            *d = (acc_dst ? *d : 0.0f) + dist_coef * sum;
        }
        return;
    }
    if (hw <= HW_DIST) return;
    float* dst = enc == 1 ? gW1 : (enc == 2 ? gW2 : gW3);
    if (!dst) return;
    float acc = 0.0f;
    for (int o = 0; o < NORD; o++) {
        const float* gr = grow + ((enc - 1) * NORD + o) * NBINS;
        const float* dt = dtab + o * 128 + 63 + m;
#pragma unroll 8
        for (int mp = 0; mp < NBINS; mp++) acc = fmaf(gr[mp], dt[-mp], acc);
    }
    float* d = dst + (size_t)hc * NBINS + m;
    *d = (acc_dst ? *d : 0.0f) + angle_coef * acc;
}
// grid: H*16 blocks.
__global__ __launch_bounds__(256) void core_gw_finish_kernel(const float* __restrict__ gwcat, int nslices, int H, int hw,
                                                             float dist_coef, float angle_coef, float ws,
                                                             float* __restrict__ gWd, float* __restrict__ gW1,
                                                             float* __restrict__ gW2, float* __restrict__ gW3) {
    core_gw_finish_block(gwcat, nslices, (size_t)H * DH * hw, hw, dist_coef, angle_coef, ws, gWd, gW1, gW2, gW3,
                         (int)blockIdx.x, false);
}

// Weight gradients of several calls of the core (the layers of a backward pass) in one launch each way.
constexpr int CORE_WG_MAX_JOBS = 8;
struct CoreWgradJob {
    const float* go;       // (N,H,16)
    const float* hist;     // (H,N,hw)
    float* gwcat;          // (nslices,H,16,hw) scratch
    float* gW[4];          // destinations (H,16,64), added to; null: not wanted
    int N, per_slice, slice0, nslices;      // atoms, atoms per slice, first slice (blockIdx.z) of this job, its slices
};
struct CoreWgradJobs {
    CoreWgradJob job[CORE_WG_MAX_JOBS];
    int njobs, H, hw;
    float dist_coef, angle_coef, ws;
    int overwrite;         // the destinations are written, not added to
};
// ---- distance window with round-to-nearest fixed-point adds ---------------------------------------------------
template <int W>
__device__ __forceinline__ void window_scatter_rn(int32_t* base, const WindowSeed& s, float cc, int wrt = 0) {
    const int Wd = W > 0 ? W : wrt, C = Wd / 2;      // (W == 0: the width is known at run time only)
    atomicAdd(base + C, rint_i(s.gc));
    float g = s.gc, r = s.rr;
#pragma unroll
    for (int m = C + 1; m < Wd; m++) { g *= r; r *= cc; atomicAdd(base + m, rint_i(g)); }
    g = s.gc; r = s.rl;
#pragma unroll
    for (int m = C - 1; m >= 0; m--) { g *= r; r *= cc; atomicAdd(base + m, rint_i(g)); }
}

// ---- shared pieces of the two main kernels ---------------------------------------------------------------------
struct CoreItem {
    Item item;
    int j0, crystal;
    bool sorted;
    int nchunks;
};
__device__ __forceinline__ CoreItem core_unpack(const CoreArgs& C, uint32_t rec, bool want_sorted) {
    CoreItem ci;
    ci.item = unpack_item(rec);
    ci.j0 = __builtin_amdgcn_readlane((int)rec, REC_J0);
    ci.crystal = __builtin_amdgcn_readlane((int)rec, REC_CRYSTAL);
    const Box& bx = ci.item.bx;
    ci.sorted = want_sorted && C.sorted_tab != nullptr && bx.R1 == C.table_R && bx.R2 == C.table_R &&
                bx.R3 == C.table_R && ci.item.a < 0.0f && C.skip_log2 > 0.0f;
    ci.nchunks = ci.sorted ? 1 : (bx.T + FC_TCAP - 1) / FC_TCAP;
    return ci;
}
// table of the item's first (or only) chunk
// build_shift_table with the rest of the last group of FC_GROUP entries filled with length +inf: a sweep then needs
// one comparison per entry, length <= limit, for "inside the table", "the row has a pair" and "within reach" together
// (the sorted tables end in such entries as well; built tables have length 0 in every real entry).
__device__ __forceinline__ void build_shift_table_padded(float4* tab, int t0, int cnt, const Box& bx, const Lattice& L,
                                                         int lane) {
    build_shift_table(tab, t0, cnt, bx, L, lane);
    const int u = cnt + lane;
    if (lane < 8 && u < ((cnt + 7) & ~7)) tab[u] = make_float4(0.f, 0.f, 0.f, __builtin_inff());
}
constexpr float FC_REACH_ALL = 3.0e38f;       // a reach that every real entry is within, and no padding entry

__device__ __forceinline__ void core_load_table(const CoreArgs& C, const CoreItem& ci, float4* tab, int lane) {
    if (ci.sorted) {
        for (int u = lane; u < FC_TCAP; u += WAVE) tab[u] = C.sorted_tab[(size_t)ci.crystal * FC_TCAP + u];
    } else if (ci.nchunks == 1) {
        build_shift_table_padded(tab, 0, ci.item.bx.T, ci.item.bx, ci.item.L, lane);
    }
}

// Operands of an item that do not depend on the item before it, fetched a whole item ahead: the two table entries
// of this lane (sorted table of the item's crystal), the lane's two query channels, and the operands of the pair
// of the first group that this lane's row serves.
struct CorePrefetch {
    float4 t0, t1;
    float2 q2;
    float rx, ry, rz;
    float2 k2, v2;
    float near;       // smallest d^2 over the images of that pair (when the batch's table of them is given)
};
__device__ __forceinline__ CorePrefetch core_prefetch(const CoreArgs& C, uint32_t rec, int it, int h, int lane) {
    CorePrefetch pf;
    pf.t0 = pf.t1 = make_float4(0.f, 0.f, 0.f, 0.f);
    pf.q2 = pf.k2 = pf.v2 = make_float2(0.f, 0.f);
    pf.rx = pf.ry = pf.rz = 0.f;
    pf.near = 3.0e38f;
    if (it < 0) return pf;
    const KernelArgs& P = C.K;
    const int H = P.H;
    const int i = __builtin_amdgcn_readlane((int)rec, REC_ATOM);
    const int e0 = __builtin_amdgcn_readlane((int)rec, REC_E0);
    const int npairs = __builtin_amdgcn_readlane((int)rec, REC_NPAIRS);
    const int j0 = __builtin_amdgcn_readlane((int)rec, REC_J0);
    const int crystal = __builtin_amdgcn_readlane((int)rec, REC_CRYSTAL);
    const int pr = lane >> 3, sub = lane & 7;
    if (C.sorted_tab) {
        const float4* src = C.sorted_tab + (size_t)crystal * FC_TCAP;
        pf.t0 = src[lane];
        pf.t1 = src[lane + WAVE];
    }
    pf.q2 = load_at<float2>(C.qs, (((uint32_t)i * (uint32_t)H + (uint32_t)h) * DH + 2u * sub) * 4u);
    if (npairs > 0) {
        // (no branch per row: a row past the end re-reads the row's last pair; nothing of it is used)
        const uint32_t el = (uint32_t)min(pr, npairs - 1);
        const uint32_t e = min((uint32_t)e0 + el, (uint32_t)(P.E - 1));
        const uint32_t jh = ((((uint32_t)j0 + el) * (uint32_t)H + (uint32_t)h) * DH + 2u * sub) * 4u;
        const float3 r3 = load_at<float3>(P.rpos, e * 12u);
        pf.rx = r3.x; pf.ry = r3.y; pf.rz = r3.z;
        pf.k2 = load_at<float2>(C.k, jh);
        pf.v2 = load_at<float2>(C.v, jh);
        if (C.pair_near) pf.near = load_at<float>(C.pair_near, e * 8u);
    }
    return pf;
}
// the item's table from what was prefetched (sorted) or built in place (one chunk)
__device__ __forceinline__ void core_store_table(const CoreItem& ci, const CorePrefetch& pf, float4* tab, int lane) {
    if (ci.sorted) {
        tab[lane] = pf.t0;
        tab[lane + WAVE] = pf.t1;
    } else if (ci.nchunks == 1) {
        build_shift_table_padded(tab, 0, ci.item.bx.T, ci.item.bx, ci.item.L, lane);
    }
}

// The record of rank r over the slow lists (list after list, a list's records in order), or -1 past the last; r is
// the same in all lanes.  Two levels, so that the wavefront waits for memory twice whatever the number of lists: every
// lane adds the counts of its own run of consecutive lists (loads that do not depend on each other), a prefix sum over
// the lanes names the run that holds rank r, and a second prefix sum over the counts of that run names the list.
struct SlowRuns { int mine, incl; };      // records of this lane's run of lists; of the runs up to and with it
__device__ __forceinline__ SlowRuns core_slow_runs(const CoreArgs& C, int lane) {
    const int n = C.slow_lists;
    const int run = (n + WAVE - 1) / WAVE;
    SlowRuns R;
    R.mine = 0;
    for (int k = 0; k < run; k++) R.mine += lane * run + k < n ? C.K.slow_count[lane * run + k] : 0;
    R.incl = wave_scan_incl(R.mine);
    return R;
}
__device__ __forceinline__ int core_slow_record(const CoreArgs& C, const SlowRuns& R, int r, int lane) {
    const int n = C.slow_lists;
    const int run = (n + WAVE - 1) / WAVE;
    if (r >= __builtin_amdgcn_readlane(R.incl, WAVE - 1)) return -1;
    const int seg = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)ballot(R.incl > r)) - 1);
    int base = __builtin_amdgcn_readlane(R.incl - R.mine, seg);
    for (int k0 = 0; k0 < run; k0 += WAVE) {
        const int li = seg * run + k0 + lane;
        const int c = (k0 + lane < run && li < n) ? C.K.slow_count[li] : 0;
        const int inc2 = wave_scan_incl(c);
        const int tot = __builtin_amdgcn_readlane(inc2, WAVE - 1);
        if (r < base + tot) {
            const int l = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)ballot(base + inc2 > r)) - 1);
            const int excl = __builtin_amdgcn_readlane(inc2 - c, l);
            return C.K.slow_list[(size_t)(seg * run + k0 + l) * C.slow_stride + (r - base - excl)];
        }
        base += tot;
    }
    return -1;
}
__device__ __forceinline__ int core_slow_record(const CoreArgs& C, int r, int lane) {
    return core_slow_record(C, core_slow_runs(C, lane), r, lane);
}
// Which record a wavefront of a main kernel starts with: the first slow_wgs wavefronts a listed one (-1: none left),
// the others the records in work order.
__device__ __forceinline__ int core_wave_record(const CoreArgs& C, int w, int lane) {
    // (the same in all lanes: said so, the index arithmetic that follows stays on the scalar unit)
    return __builtin_amdgcn_readfirstlane(w < C.slow_wgs ? core_slow_record(C, w, lane) : die_order(w - C.slow_wgs, C.K.N * C.K.H, CORE_DIE_SHIFT));
}
// The rank over the slow lists of the listed record `wid`: the counts of the lists before its own, and its place in its
// own list (records in ascending order: the entries below it).
__device__ __forceinline__ int core_slow_rank(const CoreArgs& C, int wid, int lane) {
    const int li = wid / C.slow_stride;
    int part = 0;
    for (int c0 = lane; c0 < li; c0 += WAVE) part += C.K.slow_count[c0];
    const int n = C.K.slow_count[li];
    const int32_t* lst = C.K.slow_list + (size_t)li * C.slow_stride;
    for (int k = lane; k < n; k += WAVE) part += lst[k] < wid ? 1 : 0;
    return __builtin_amdgcn_readlane(wave_scan_incl(part), WAVE - 1);
}
// A listed record is left to the leading wavefront of its rank; ranks past the leading wavefronts stay in place.
__device__ __forceinline__ bool core_record_taken_elsewhere(const CoreArgs& C, uint32_t rec, int wid, int lane) {
    if (C.slow_wgs == 0 || (int)(blockIdx.x * CORE_WPB + (threadIdx.x >> 6)) < C.slow_wgs) return false;
    if (((uint32_t)__builtin_amdgcn_readlane((int)rec, REC_BOX) & C.slow_flag) == 0u) return false;
    return core_slow_rank(C, wid, lane) < C.slow_wgs;
}

// =================================================================================================================
// forward
// =================================================================================================================
// The distance bins of an item exist COPIES times in LDS, a copy per value of the lane's lowest bits, where there are many items:
// most images of an item lie at nearly the same distance, a few bins of 64, and the lanes of an atomic instruction that meet on
// a word go one after the other (inference of 180 224 items, 64 angle bins: LDS busy for 134 M clocks, 72 M of them such waits;
// distances alone 78 M and 37 M).  4096 crystals, four layers, in us: 64 angle bins 1 copy 2650, 2 copies 2588, 4 (less LDS for
// other wavefronts) 2655; distances alone, four heads per wavefront, 1173, -, 1030.  Rows of 40 to 200 pairs in
// training lose 0.6 % with 2 copies, few items (item_pass_kernel) 0.5 to 1.3 %.
constexpr int DIST_STRIDE = NBINS + 8;      // words from one copy to the next: other banks
// An item's histogram in LDS: its words, then the further copies of its distance bins.
template <int ANG, bool LEAN, int COPIES>
struct CoreHist {
    static constexpr int WORDS = LEAN && ANG == NBINS ? core_hist_words(ANG, LEAN) : core_hist_lds_words(ANG);
    static constexpr int FIRST = WORDS + 8;      // (other banks than copy 0)
    static constexpr int ALL = COPIES > 1 ? FIRST + (COPIES - 1) * DIST_STRIDE : WORDS;
    static_assert(WORDS % 4 == 0 && ALL % 4 == 0 && (COPIES & (COPIES - 1)) == 0, "");
    static constexpr __host__ __device__ int copy(int c) { return c == 0 ? 0 : FIRST + (c - 1) * DIST_STRIDE; }
    // first word of the distance bins that this lane adds to
    static __device__ __forceinline__ int dist_word(int lane) {
        const int c = lane & (COPIES - 1);
        return COPIES > 1 && c > 0 ? FIRST + (c - 1) * DIST_STRIDE : 0;
    }
    // word / four words with the copies of the distance bins added
    static __device__ __forceinline__ int word(const int32_t* hist, int w) {
        int v = hist[w];
        if (COPIES > 1 && w < NBINS) {
#pragma unroll
            for (int c = 1; c < COPIES; c++) v += hist[copy(c) + w];
        }
        return v;
    }
    static __device__ __forceinline__ int4 word4(const int32_t* hist, int u) {
        int4 v = reinterpret_cast<const int4*>(hist)[u];
        if (COPIES > 1 && u < NBINS / 4) {
#pragma unroll
            for (int c = 1; c < COPIES; c++) {
                const int4 w = reinterpret_cast<const int4*>(hist + copy(c))[u];
                v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
            }
        }
        return v;
    }
    static __device__ __forceinline__ void clear(int32_t* hist, int lane) {
#pragma unroll
        for (int u = 0; u < (ALL / 4 + WAVE - 1) / WAVE; u++)
            if (ALL % (4 * WAVE) == 0 || lane + WAVE * u < ALL / 4) reinterpret_cast<int4*>(hist)[lane + WAVE * u] = make_int4(0, 0, 0, 0);
    }
    // times fac, rounded once per word: the copies are added up first
    static __device__ __forceinline__ void rescale(int32_t* hist, float fac, int lane) {
        constexpr int NU = (WORDS / 4 + WAVE - 1) / WAVE;
        int4 v[NU];
#pragma unroll
        for (int u = 0; u < NU; u++)
            if (WORDS % (4 * WAVE) == 0 || lane + WAVE * u < WORDS / 4) v[u] = word4(hist, lane + WAVE * u);
        if (COPIES > 1 && lane < NBINS / 4) {
#pragma unroll
            for (int c = 1; c < COPIES; c++) reinterpret_cast<int4*>(hist + copy(c))[lane] = make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < NU; u++)
            if (WORDS % (4 * WAVE) == 0 || lane + WAVE * u < WORDS / 4) reinterpret_cast<int4*>(hist)[lane + WAVE * u] =
                make_int4(rint_i((float)v[u].x * fac), rint_i((float)v[u].y * fac), rint_i((float)v[u].z * fac), rint_i((float)v[u].w * fac));
    }
};
template <int HWK, int NLOGIT>
struct CoreFwdShared {
    float4 tab[FC_TCAP];
    uint16_t list[FC_LISTCAP];
    __attribute__((aligned(16))) int32_t hist[HWK];
    float4 pairA[FC_GROUP];      // rx, ry, rz, d2min
    float pairC[FC_GROUP];       // exp(logit - running max) / S in fixed-point units
    float logit_s[NLOGIT];       // logits of the row (rows of more pairs park them in the probability array)
};
// LEAN: inference, nothing is kept for a backward pass: fewer nodes for the moments; z and the probabilities are not written.
template <int ANG, bool LEAN, int COPIES = 1>
using CoreFwdLds = CoreFwdShared<CoreHist<ANG, LEAN, COPIES>::ALL, LEAN ? 4 : FC_LOGCAP>;
// Sums of 4 values over the lanes of a wavefront: lane l gets the sum of value l / 16.
__device__ __forceinline__ float wave_sum4(const float (&v)[4], int lane) {
    // each step halves the values a lane holds: it keeps one half and hands its partner the other
    const bool b5 = (lane & 32) != 0, b4 = (lane & 16) != 0;
    const float p = (b5 ? v[2] : v[0]) + __shfl_xor(b5 ? v[0] : v[2], 32), q = (b5 ? v[3] : v[1]) + __shfl_xor(b5 ? v[1] : v[3], 32);
    float s = (b4 ? q : p) + __shfl_xor(b4 ? p : q, 16);
    s += dpp_move<0xB1>(s); s += dpp_move<0x4E>(s); s += dpp_move<0x141>(s);
    return s + dpp_move<0x128>(s);
}
// ---- products with the weights -----------------------------------------------------------------------------------
// out (N,H,16) += Wcat_h (16, hw) . hist: sixteen items of a head through MFMA 16x16x4, the sum over the words in slices
// that are added in a fixed order (256 words per slice with all moments, 144 with the nodes of inference), whichever
// wavefront makes them: the result depends neither on timing nor on which of the two places below makes it.
//   core_project_done     in the main kernel, by the wavefront that completes the sixteen;
//   core_project_kernel   in a launch of its own, a workgroup per sixteen, a wavefront per slice.
// The launch is bound by reading the histograms back: 519 MB (22 528 atoms, 720 words) in 131 us (4.0 TB/s).
template <int HWK> struct ProjectSlices;
template <> struct ProjectSlices<HW_ANG> { static constexpr int N = 4, UNITS = 16, BATCH = 8; };
template <> struct ProjectSlices<HW_LEAN> { static constexpr int N = 5, UNITS = 9, BATCH = 5; };
template <> struct ProjectSlices<HW_ANG16> { static constexpr int N = 2, UNITS = 4, BATCH = 4; };
template <> struct ProjectSlices<HW_DIST> { static constexpr int N = 1, UNITS = 4, BATCH = 4; };
// A slice: UNITS x 16 words, BATCH units' loads in flight together.  a(u): the four words of this lane's row of unit u; bp: its
// weights.  The four lanes of a row read 64 consecutive bytes per load; which word of the sum a lane holds does not matter as
// long as both operands agree.
template <int UNITS, int BATCH, typename Load>
__device__ __forceinline__ v4f_c project_slice(Load&& a, const float4* bp) {
    v4f_c acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u0 = 0; u0 < UNITS; u0 += BATCH) {
        float4 a4[BATCH], b4[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++)
            if (u0 + u < UNITS) { a4[u] = a(u0 + u); b4[u] = bp[4 * (u0 + u)]; }
        __builtin_amdgcn_sched_barrier(0);         // (all loads in flight before the first product)
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            if (u0 + u >= UNITS) continue;
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[u].x, b4[u].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[u].y, b4[u].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[u].z, b4[u].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[u].w, b4[u].w, acc, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}

// What wavefronts of other compute units and dies read in the same launch is written, and read, at device scope: the store goes
// through to the memory behind the dies' L2s, the load takes nothing that an L1 or another die's L2 holds from before.  With
// s_waitcnt between a wavefront's stores and its ticket, and a ticket that is drawn at device scope, whoever draws the last of
// sixteen tickets reads what the other fifteen wrote; no cache is written back or emptied as a whole, which a fence of that
// scope does (199 us for a launch of 2372 atoms' weight gradients with a fence before every ticket).
constexpr int CPOL_DEVICE = 16;      // sc1
typedef int v4i_c __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t device_rsrc(float* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ float4 load_device4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const v4i_c v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, CPOL_DEVICE);
    return make_float4(__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z), __int_as_float(v.w));
}
__device__ __forceinline__ void store_device4(__amdgpu_buffer_rsrc_t r, uint32_t off, float4 v) {
    const v4i_c w = {__float_as_int(v.x), __float_as_int(v.y), __float_as_int(v.z), __float_as_int(v.w)};
    __builtin_amdgcn_raw_buffer_store_b128(w, r, (int)off, 0, CPOL_DEVICE);
}
__device__ __forceinline__ void store_device(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A lane's row of the histograms and the atom it belongs to: rank (lane & 15) of the sixteen.  (A rank past the last member
// takes the last.)
struct ProjectRow { int atom; uint32_t row; };
__device__ __forceinline__ ProjectRow project_row(const uint32_t* records, int sixteen, int members, int h, int H, int lane) {
    const int rank = min(lane & 15, members - 1);
    ProjectRow R;
    R.atom = (int)records[((size_t)sixteen_place(sixteen, rank) * H + h) * REC_WORDS + REC_ATOM];
    R.row = (uint32_t)(sixteen * 16 + rank);
    return R;
}
// Rows of a head's histograms where they lie in the order of the sixteens.
__host__ __device__ constexpr int project_rows(int N) { return 16 * sixteens(N); }

// Inference of many items with the angle encoding: the item of this wavefront is done, its histogram row and its part of `out`
// stored at device scope.  Draws the ticket of its sixteen; whoever draws the last one makes their products.  What is read so is
// still in the dies' memory-side cache, and the product's 180 matrix instructions run beside the other wavefronts' vector ones: 22 528
// atoms at 64 bins main kernel 393 us + products 131 in a launch of their own -> 449 + 30 (the last fifth, see products_in_place).
// Sixteen items of ONE die: were they dealt over the dies, the one that happens to be behind would draw the last ticket of
// nearly all, make the products alone and fall further behind (seven dies done after 416 us, the eighth after 1085).
// Training, whose rows have 1024 words in the order of the atoms, keeps the launch: 18 976 items 80 us in two launches, 84 so.
template <int HWK>
__device__ __forceinline__ void core_project_done(const CoreArgs& C, int it, int h, int lane) {
    using S = ProjectSlices<HWK>;
    const int H = C.K.H, N = C.K.N, sixteen = sixteen_of(it), members = sixteen_members(sixteen, N);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int ticket = 0;
    if (lane == 0)
        ticket = __hip_atomic_fetch_add(C.tickets + (sixteen * H + h) * TICKET_STRIDE, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(ticket) != members - 1) return;
    asm volatile("" ::: "memory");
    const int col = lane & 15, kk = lane >> 4, rows = project_rows(N);
    const ProjectRow R = project_row(C.K.items, sixteen, members, h, H, lane);
    const __amdgpu_buffer_rsrc_t hist = device_rsrc(C.hist + (size_t)h * rows * HWK, (uint32_t)rows * (HWK * 4u));
    uint32_t aoff = (R.row * HWK + 4u * kk) * 4u;
    const float4* bp = reinterpret_cast<const float4*>(C.wcat + ((size_t)h * DH + col) * HWK) + kk;
    v4f_c sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < S::N; s++) {
        const v4f_c acc = project_slice<S::UNITS, S::BATCH>([&](int u) { return load_device4(hist, aoff + 64u * u); }, bp);
        if (s == 0) sum = acc;
        else sum += acc;
        aoff += 64u * S::UNITS;
        bp += 4 * S::UNITS;
    }
    // component r of lane (kk, col): rank 4 kk + r, channel col
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float* dst = C.out + ((size_t)__shfl(R.atom, 4 * kk + r) * H + h) * DH + col;
        const float own = __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (4 * kk + r < members) *dst = own + sum[r];
    }
}

// ANG: angle bins, 0 (distance encoding alone), 64 (moment series) or 16 (basis values added directly)
// wid: this wavefront's (item, head)
// wcat: not null: the wavefront makes the product of its histogram with the head's weights itself, the histogram stays in
// LDS (LEAN only)
// own: not null: the item's record and first operands, in registers
// given: the item is this wavefront's, listed or not
struct CoreOwn { uint32_t rec; CorePrefetch pf; };
// HAND_OVER (LEAN only): the histogram stays in LDS as float32 words, with the item's part of `out` and its atom in front of the
// table, for other wavefronts of the workgroup (CoreProductWeights), which wait at a barrier until it is there
template <int WL, int ANG, bool COS_ABS, bool LEAN, int COPIES = 1, bool HAND_OVER = false>
__device__ __forceinline__ void fused_core_fwd_body(const CoreArgs& C, CoreFwdLds<ANG, LEAN, COPIES>& sh, int wid,
                                                    const float* __restrict__ wcat = nullptr, const CoreOwn* own = nullptr,
                                                    bool given = false) {
    constexpr bool HAS_ANG = ANG > 0;
    constexpr int HWK = core_hist_words(ANG, LEAN);          // words per item in memory
    using Hist = CoreHist<ANG, LEAN, COPIES>;
    constexpr int HWL = Hist::WORDS;                         // ... and in LDS
    constexpr int NODES = LEAN ? LEAN_NODES : NBINS;
    constexpr bool VEC = HWL == HWK && HWK >= 4 * WAVE;      // clear, rescale and store four words per lane at a time
    constexpr int NW = VEC ? (HWK / 4 + WAVE - 1) / WAVE : 1;
    constexpr bool FULL = HWK % (4 * WAVE) == 0;
    constexpr bool PLACES = LEAN && HAS_ANG;                 // histograms in the order of the sixteens
    float4* const tab = sh.tab;
    uint16_t* const list = sh.list;
    int32_t* const hist = sh.hist;
    float4* const pairA = sh.pairA;
    float* const pairC = sh.pairC;
    float* const logit_s = sh.logit_s;

    const KernelArgs& P = C.K;
    const int lane = threadIdx.x & (WAVE - 1);
    const int H = P.H;
    const int it_cur = div_heads(P, wid);      // items in descending order of their pair count: the long ones start first
    const int h = wid - it_cur * H;
    const int pr = lane >> 3;          // pair of the group served by this 8-lane row
    const int sub = lane & 7;          // position in the row
    const BasisConsts bc = P.bc;
    const int WLr = WL > 0 ? WL : bc.len_window;      // bins of the distance window (WL == 0: known at run time only)
    const float prune = (P.prune_log2 > 0.0f) ? -P.prune_log2 : -3.0e38f;
    const float INF = __builtin_inff();

    if (it_cur >= P.N) return;
    Hist::clear(hist, lane);
    const int dist0 = Hist::dist_word(lane);
    wave_sync();

    CFH_PH_DECL
    {
        const uint32_t rec_cur = own ? own->rec : load_record_lane(P, it_cur, h, lane);
        if (!own && !given && core_record_taken_elsewhere(C, rec_cur, wid, lane)) return;
        const CorePrefetch pf = own ? own->pf : core_prefetch(C, rec_cur, it_cur, h, lane);
        CFH_PH(0);
        const CoreItem ci = core_unpack(C, rec_cur, true);
        const int i = ci.item.i;
        const float a = ci.item.a;
        const float a2 = a * LOG2E;
        const Lattice L = ci.item.L;
        const Box bx = ci.item.bx;
        const bool sorted = ci.sorted;
        const int nchunks = ci.nchunks;
        float f[3][3];
        if (HAS_ANG) {
#pragma unroll
            for (int ax = 0; ax < 3; ax++)
#pragma unroll
                for (int d = 0; d < 3; d++) f[ax][d] = rec_f(rec_cur, REC_FRAMES + ax * 3 + d);
        }
        const int e0 = ci.item.e0, npairs = ci.item.npairs;
        wave_sync();                          // the previous item's readers of the table are done
        core_store_table(ci, pf, tab, lane);
        wave_sync();
        const size_t ih = (size_t)i * H + h;
        const float2 q2 = pf.q2;
        // 2^30 / npairs: sums of weights <= 1 each fit (hardware reciprocal: any scale near it will do, the histogram
        // is divided by the same number when it is written)
        const float fixs = 1073741824.0f * hw_rcp((float)max(npairs, 1));
        const float cutS = (C.skip_log2 > 0.0f && a2 < 0.0f) ? C.skip_log2 * hw_rcp(-a2) : INF;      // (a bound with margins)
        float m_run = -INF;                   // running maximum of the logits (wave-uniform)
        float Dl = 0.0f;                      // this lane's share of the softmax denominator
        float2 accv = make_float2(0.f, 0.f);  // sum_j exp(logit_j - m_run) v_j, channels 2 sub, 2 sub + 1
        unsigned long long n_eval = 0, n_seen = 0;      // wave-uniform counts

        // operands of the pair served by this row, fetched one group ahead (the first group: with the item)
        float nrx = pf.rx, nry = pf.ry, nrz = pf.rz, nnear = pf.near;
        float2 nk2 = pf.k2, nv2 = pf.v2;
        // The nearest image of every pair over the usual box comes with the batch.  An item whose box CONTAINS the usual
        // one takes it as the reference of its weights as well (any reference gives the same normalised weights and
        // the same z; only the pruning threshold moves with it, should an image outside the usual box be nearer)
        const bool contains_usual = C.sorted_tab != nullptr && bx.R1 >= C.table_R && bx.R2 >= C.table_R && bx.R3 >= C.table_R;
        const bool near_known = (sorted || contains_usual) && C.pair_near != nullptr;
        // several chunks: the survivors of all chunks go into one list with their index in the whole box, and the
        // heavy pass makes their shifts from that index instead of reading a table: one sweep, each chunk built once
        const bool one_list = nchunks > 1 && bx.T <= FC_BIGT;
        auto fetch = [&](int g0) {
            // (no branch per row: a row past the end re-reads the row's last pair; nothing of it is used)
            const uint32_t el = (uint32_t)min(g0 + pr, npairs - 1);
            const uint32_t e = min((uint32_t)e0 + el, (uint32_t)(P.E - 1));
            const uint32_t jh = ((((uint32_t)ci.j0 + el) * (uint32_t)H + (uint32_t)h) * DH + 2u * sub) * 4u;
            const float3 r3 = load_at<float3>(P.rpos, e * 12u);
            nrx = r3.x; nry = r3.y; nrz = r3.z;
            nk2 = load_at<float2>(C.k, jh);
            nv2 = load_at<float2>(C.v, jh);
            if (near_known) nnear = load_at<float>(C.pair_near, e * 8u);
        };

        // one sweep of this row's pair over the table(s): fn(inside, index in the chunk, first index of the chunk, d^2, rows inside)
        auto sweep = [&](bool active, float rx, float ry, float rz, float reach, auto&& fn) {
            const float lim = active ? fminf(reach, FC_REACH_ALL) : -1.0f;      // (lengths are >= 0; padding: +inf)
            for (int ch = 0; ch < nchunks; ch++) {
                const int t0c = ch * FC_TCAP;
                const int cnt = sorted ? bx.T : min(FC_TCAP, bx.T - t0c);
                if (nchunks > 1) {
                    wave_sync();
                    build_shift_table_padded(tab, t0c, cnt, bx, L, lane);
                    wave_sync();
                }
                float4 v = tab[sub];
                for (int t0 = 0; t0 < cnt; t0 += FC_GROUP) {
                    const int t = t0 + sub;
                    const float4 vn = tab[min(t + FC_GROUP, FC_TCAP - 1)];      // the next step's entry, in flight meanwhile
                    const bool in = v.w <= lim;
                    const uint64_t inm = ballot(in);
                    if (sorted && inm == 0) break;               // every row is past its reach (lengths ascend)
                    const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
                    fn(in, t, t0c, fmaf(dx, dx, fmaf(dy, dy, dz * dz)), __popcll(inm));
                    v = vn;
                }
            }
        };

        // scatter of the current list (entries point into the resident table)
        auto heavy_impl = [&](int nlist, auto big) {
            constexpr bool BIG = decltype(big)::value;      // entries (pair << FC_BIGSHIFT | index in the box), no table
            // (hardware reciprocals, within an ulp: the quotients below stay exact all the same)
            const float inv_s3 = BIG ? hw_rcp((float)bx.s3) : 0.0f, inv_s2 = BIG ? hw_rcp((float)bx.s2) : 0.0f;
            for (int base = 0; base < nlist; base += WAVE) {
                const int idx = base + lane;
                if (idx < nlist) {
                    const uint32_t ent = list[idx];
                    const int pp = BIG ? (int)(ent >> FC_BIGSHIFT) : (int)(ent >> FC_SHIFT);
                    float4 v;
                    if (BIG) {
                        const int tg = (int)(ent & (FC_BIGT - 1));
                        // (exact: the quotients stay below 2^13 and the fractions at least 1 / (2 s) from an integer)
                        const int q = (int)(((float)tg + 0.5f) * inv_s3), i3 = tg - q * bx.s3;
                        const int i1 = (int)(((float)q + 0.5f) * inv_s2), i2 = q - i1 * bx.s2;
                        const float n1 = (float)(i1 - bx.R1), n2 = (float)(i2 - bx.R2), n3 = (float)(i3 - bx.R3);
                        v.x = fmaf(L.t[6], n3, fmaf(L.t[3], n2, L.t[0] * n1));      // as build_shift_table makes them
                        v.y = fmaf(L.t[7], n3, fmaf(L.t[4], n2, L.t[1] * n1));
                        v.z = fmaf(L.t[8], n3, fmaf(L.t[5], n2, L.t[2] * n1));
                        v.w = 0.0f;
                    } else {
                        v = tab[ent & (FC_TCAP - 1)];
                    }
                    const float4 pa = pairA[pp];
                    const float dx = pa.x + v.x, dy = pa.y + v.y, dz = pa.z + v.z;
                    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    const float w = hw_exp2(a2 * (d2 - pa.w)) * pairC[pp];
                    {
                        const float d = hw_sqrt(d2);
                        const float u = d * bc.inv_interval;
                        int start = (int)(u - bc.start_off);          // truncation toward zero
                        start = max(0, min(start, NBINS - WLr));
                        const float beta_c = ((float)(start + WLr / 2 + 1) - u) * bc.len_step;
                        const WindowSeed s = window_seed(beta_c, bc.len_step, w);
                        window_scatter_rn<WL>(hist + dist0 + start, s, bc.len_cc, WLr);
                    }
                    if (HAS_ANG) {
                        if (d2 > 1e-5f) {       // the self image contributes to S and the distance encoding only
                            const float rinv = hw_rsq(d2);
#pragma unroll
                            for (int ax = 0; ax < 3; ax++) {
                                float cs = (dx * f[ax][0] + dy * f[ax][1] + dz * f[ax][2]) * rinv;
                                if (COS_ABS) cs = fabsf(cs);
                                const float uu = (cs - bc.ang_mu0) * bc.ang_inv_interval;      // in bin (LEAN: node) units
                                if (ANG == SMALL_A) {
                                    // all 16 basis values, outwards from bin 8 by the two-sided recurrence (sigma >= 1
                                    // bin: the value at bin 8 is at least e^-32 of the peak, no underflow)
                                    const WindowSeed sa = window_seed(((float)(SMALL_A / 2) - uu) * bc.ang_step, bc.ang_step, w);
                                    window_scatter_rn<SMALL_A>(hist + HW_DIST + (lane & (A16_COPIES - 1)) * A16_STRIDE + ax * SMALL_A,
                                                               sa, bc.ang_cc);
                                    continue;
                                }
                                const float mf = clampf(__builtin_rintf(uu), 0.0f, (float)(NODES - 1));
                                const float eps = 2.0f * (uu - mf);
                                int32_t* hb = hist + HW_DIST + ax * NORD * NODES + (int)mf;
                                float val = w;
                                atomicAdd(hb, rint_i(val));
#pragma unroll
                                for (int o = 1; o < NORD; o++) { val *= eps; atomicAdd(hb + o * NODES, rint_i(val)); }
                            }
                        }
                    }
                }
            }
            n_eval += (unsigned long long)nlist;
        };
        auto heavy = [&](int nlist) { heavy_impl(nlist, std::false_type{}); };

        for (int g0 = 0; g0 < npairs; g0 += FC_GROUP) {
            const float rx = nrx, ry = nry, rz = nrz;
            const float2 k2 = nk2, v2 = nv2;
            float d2min = nnear;
            if (g0 + FC_GROUP < npairs) fetch(g0 + FC_GROUP);
            const bool active = g0 + pr < npairs;
            const float rn = hw_sqrt(fmaf(rx, rx, fmaf(ry, ry, rz * rz)));

            float Sb, S;
            int nlist;
            bool spilled;                     // (several chunks) more survivors than the list holds: the chunks again, one by one
            bool known = near_known;
            for (;;) {
            // ---- pass A: nearest image (known beforehand for the usual box)
            CFH_PH(1);
            if (!known) {
                d2min = 3.0e38f;
                sweep(active, rx, ry, rz, sorted ? fmaf(2.0002f, rn, 1e-4f) : FC_REACH_ALL,
                      [&](bool in, int, int, float d2, int cnt_in) { d2min = in ? fminf(d2min, d2) : d2min; n_seen += cnt_in; });
                d2min = half_min(d2min);
            }

            // ---- pass B: weights, normaliser and (one-chunk tables) the survivors
            CFH_PH(2);
            const float reachB = sorted ? fmaf(1.0001f, rn + hw_sqrt(d2min + cutS), 1e-4f) : FC_REACH_ALL;
            Sb = 0.0f;
            nlist = 0;
            spilled = false;
            if (nchunks == 1) {
                sweep(active, rx, ry, rz, reachB, [&](bool in, int t, int, float d2, int cnt_in) {
                    const float ex = in ? a2 * (d2 - d2min) : -INF;      // (2^-inf = 0, and -inf is below every threshold)
                    Sb += hw_exp2(ex);
                    n_seen += cnt_in;
                    const bool keep = ex >= prune;
                    const uint64_t m = ballot(keep);
                    if (keep) list[nlist + lane_prefix(m)] = (uint16_t)((pr << FC_SHIFT) | t);
                    nlist += __popcll(m);
                });
            } else {
                sweep(active, rx, ry, rz, reachB, [&](bool in, int t, int t0c, float d2, int cnt_in) {
                    const float ex = in ? a2 * (d2 - d2min) : -INF;
                    Sb += hw_exp2(ex);
                    n_seen += cnt_in;
                    if (one_list && !spilled) {
                        const bool keep = ex >= prune;
                        const uint64_t m = ballot(keep);
                        if (nlist + __popcll(m) > FC_LISTCAP) spilled = true;
                        else {
                            if (keep) list[nlist + lane_prefix(m)] = (uint16_t)((pr << FC_BIGSHIFT) | (t0c + t));
                            nlist += __popcll(m);
                        }
                    }
                });
            }
            S = half_sum(Sb);
            // a reference borrowed from the usual box may lie far above the nearest image of a larger box (a strongly
            // sheared cell): a sum of weights of 2^24 and more says so (with the nearest image as the reference it is at
            // most the number of translations, 2^13), and the group is done again with a sweep for the nearest
            if (known && !sorted && ballot(active && !(S < 0x1p24f)) != 0) { known = false; continue; }
            break;
            }

            // ---- logits, running softmax
            CFH_PH(3);
            const float qk = half_sum(fmaf(q2.x, k2.x, q2.y * k2.y));
            const float z = fmaf(hw_log2(S), LN2, a * d2min);
            const float logit = active ? qk + z : -INF;
            const float gmax = uniform_f(wave_maxf(logit));
            if (gmax > m_run) {
                if (m_run > -INF) {
                    const float fac = hw_exp2((m_run - gmax) * LOG2E);
                    Hist::rescale(hist, fac, lane);
                    accv.x *= fac; accv.y *= fac; Dl *= fac;
                }
                m_run = gmax;
            }
            const float ew = active ? hw_exp2((logit - m_run) * LOG2E) : 0.0f;
            accv.x = fmaf(ew, v2.x, accv.x);
            accv.y = fmaf(ew, v2.y, accv.y);
            if (sub == 0 && active) {
                const uint32_t eh = ((uint32_t)(e0 + g0 + pr) * (uint32_t)H + (uint32_t)h) * 4u;      // byte offset
                pairA[pr] = make_float4(rx, ry, rz, d2min);
                pairC[pr] = ew * hw_rcp(S) * fixs;
                if (!LEAN) *reinterpret_cast<float*>(reinterpret_cast<char*>(C.z) + eh) = z;
                if (LEAN) {}
                else if (npairs <= FC_LOGCAP) logit_s[g0 + pr] = logit;
                else *reinterpret_cast<float*>(reinterpret_cast<char*>(C.prob) + eh) = logit;      // the logit for now; normalised when the row is complete
                Dl += ew;
            }
            wave_sync();

            // ---- heavy pass
            CFH_PH(4);
            if (nchunks == 1) heavy(nlist);
            else if (one_list && !spilled) heavy_impl(nlist, std::true_type{});
            else {
                for (int ch = 0; ch < nchunks; ch++) {
                    const int t0c = ch * FC_TCAP;
                    const int cnt = min(FC_TCAP, bx.T - t0c);
                    wave_sync();
                    build_shift_table(tab, t0c, cnt, bx, L, lane);
                    wave_sync();
                    int nl = 0;
                    for (int t0 = 0; t0 < cnt; t0 += FC_GROUP) {
                        const int t = t0 + sub;
                        const float4 v = tab[min(t, cnt - 1)];
                        const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
                        const float ex = a2 * (fmaf(dx, dx, fmaf(dy, dy, dz * dz)) - d2min);
                        const bool keep = active && t < cnt && ex >= prune;
                        const uint64_t m = ballot(keep);
                        if (keep) list[nl + lane_prefix(m)] = (uint16_t)((pr << FC_SHIFT) | t);
                        nl += __popcll(m);
                    }
                    wave_sync();
                    heavy(nl);
                }
            }
            wave_sync();                      // list, pair data and (several chunks) the table may be rewritten
            CFH_PH(3);
        }

        // ---- the row is complete: normalise and write
        CFH_PH(7);
        auto count_item = [&] {
            CFH_PH_FLUSH(P.stats);
            if (P.stats && lane == 0) {
                atomicAdd(P.stats + STAT_FWD_EVAL, n_eval);
                atomicAdd(P.stats + STAT_FWD_RAW, (unsigned long long)bx.T * (unsigned long long)npairs);
                atomicAdd(P.stats + STAT_FWD_PAIRS, (unsigned long long)npairs);
                atomicAdd(P.stats + STAT_FWD_SEEN, n_seen);
            }
        };
        const float D = uniform_f(wave_sum(Dl));
        const float inv = D > 0.0f ? hw_rcp(D) : 0.0f;
        const float sc = inv * hw_rcp(fixs);
        if (LEAN && (HAND_OVER || wcat)) {
            // Four words per lane at a time (fewer words: one).  A loop over the channels, four at a time with their loads in
            // flight together: a wavefront runs through this once, and fetching the instructions of all sixteen took longer than
            // the loop's waits for weights (a layer's launch of 64 items 20.0 us, in the loop 18.2; whole calls of 4872 items 272 and
            // 250 us).  The loads of eight channels together: 136 registers, three wavefronts per SIMD.
            constexpr int NV = VEC ? 4 * NW : HWK / WAVE;
            float word[NV];
            if (VEC) {
#pragma unroll
                for (int u = 0; u < NW; u++) {
                    int4 hv = make_int4(0, 0, 0, 0);
                    if (FULL || lane + WAVE * u < HWL / 4) hv = Hist::word4(hist, lane + WAVE * u);
                    word[4 * u] = (float)hv.x * sc; word[(4 * u + 1) % NV] = (float)hv.y * sc;
                    word[(4 * u + 2) % NV] = (float)hv.z * sc; word[(4 * u + 3) % NV] = (float)hv.w * sc;
                }
            } else {
#pragma unroll
                for (int u = 0; u < NV; u++) {
                    const int w = lane + WAVE * u;
                    int32_t sum = 0;
                    if (ANG != SMALL_A || w < HW_DIST) sum = Hist::word(hist, w);
                    else if (w < HW_DIST + 3 * SMALL_A) {
#pragma unroll
                        for (int c = 0; c < A16_COPIES; c++) sum += hist[HW_DIST + c * A16_STRIDE + (w - HW_DIST)];
                    }
                    word[u] = (float)sum * sc;
                }
            }
            const float ox = rows8_sum(accv.x) * inv, oy = rows8_sum(accv.y) * inv;      // (the same in every 8-lane row)
            if (HAND_OVER) {
                wave_sync();
#pragma unroll
                for (int u = 0; u < NV; u++) {
                    const int w = VEC ? 4 * (lane + WAVE * (u >> 2)) + (u & 3) : lane + WAVE * u;
                    if (w < HWK) hist[w] = __float_as_int(word[u]);
                }
                if (lane < FC_GROUP) reinterpret_cast<float2*>(tab)[lane] = make_float2(ox, oy);
                if (lane == 0) tab[4].x = __int_as_float(i);
                __syncthreads();      // (the statistics wait, not the product)
                count_item();
                return;
            }
            const float* Wh = wcat + (size_t)h * DH * HWK;
            float* const dst = C.out + ih * DH;
#pragma unroll 1
            for (int c0 = 0; c0 < DH; c0 += 4, Wh += 4 * HWK) {
                float v[4];
#pragma unroll
                for (int c = 0; c < 4; c++) v[c] = lane == ((c0 + c) >> 1) ? ((c & 1) ? oy : ox) : 0.0f;
                if (VEC) {
                    float4 wt[4][NW];
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int u = 0; u < NW; u++)      // (a lane past the end reads the last words; its own are zero)
                            wt[c][u] = *reinterpret_cast<const float4*>(Wh + c * HWK + 4 * min(lane + WAVE * u, HWK / 4 - 1));
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int u = 0; u < NW; u++)
                            v[c] = fmaf(word[4 * u], wt[c][u].x, fmaf(word[(4 * u + 1) % NV], wt[c][u].y,
                                   fmaf(word[(4 * u + 2) % NV], wt[c][u].z, fmaf(word[(4 * u + 3) % NV], wt[c][u].w, v[c]))));
                } else {
                    float wt[4][NV];
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int u = 0; u < NV; u++) wt[c][u] = Wh[c * HWK + lane + WAVE * u];
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int u = 0; u < NV; u++) v[c] = fmaf(word[u], wt[c][u], v[c]);
                }
                const float sum = wave_sum4(v, lane);
                if ((lane & 15) == 0) dst[c0 + (lane >> 4)] = sum;
            }
        } else {
            const float ox = rows8_sum(accv.x) * inv, oy = rows8_sum(accv.y) * inv;
            if (lane < FC_GROUP) {
                if (PLACES) { store_device(C.out + ih * DH + 2 * sub, ox); store_device(C.out + ih * DH + 2 * sub + 1, oy); }
                else *reinterpret_cast<float2*>(C.out + ih * DH + 2 * sub) = make_float2(ox, oy);
            }
        }
        if (!(LEAN && wcat)) {
            // all reads first (one LDS round trip instead of one per word), then store; a lane takes four
            // consecutive words at a time
            // head-major: the rows of a head are contiguous
            float* dst = C.hist + (PLACES ? (size_t)h * project_rows(P.N) + sixteen_of(it_cur) * 16 + sixteen_rank(it_cur)
                                          : (size_t)h * P.N + i) * HWK;
            if (ANG == SMALL_A) {
                // distance bins as they are, every angle bin as the sum of its copies (integers: any order), zeros behind
                for (int u = lane; u < HWK; u += WAVE) {
                    int32_t sum = 0;
                    if (u < HW_DIST) sum = Hist::word(hist, u);
                    else if (u < HW_DIST + 3 * SMALL_A) {
#pragma unroll
                        for (int c = 0; c < A16_COPIES; c++) sum += hist[HW_DIST + c * A16_STRIDE + (u - HW_DIST)];
                    }
                    if (PLACES) store_device(dst + u, (float)sum * sc);
                    else dst[u] = (float)sum * sc;
                }
            } else if (VEC) {
                int4 hv[NW];
#pragma unroll
                for (int u = 0; u < NW; u++)
                    if (FULL || lane + WAVE * u < HWL / 4) hv[u] = Hist::word4(hist, lane + WAVE * u);
                const __amdgpu_buffer_rsrc_t words = device_rsrc(dst, HWK * 4u);
#pragma unroll
                for (int u = 0; u < NW; u++)
                    if (FULL || lane + WAVE * u < HWL / 4) {
                        const float4 v = make_float4((float)hv[u].x * sc, (float)hv[u].y * sc, (float)hv[u].z * sc, (float)hv[u].w * sc);
                        if (PLACES) store_device4(words, 16u * (lane + WAVE * u), v);
                        else reinterpret_cast<float4*>(dst)[lane + WAVE * u] = v;
                    }
            } else {
                for (int u = lane; u < HWK; u += WAVE) dst[u] = (float)Hist::word(hist, u) * sc;
            }
        }
        if (LEAN) {}
        else if (npairs <= FC_LOGCAP) {                          // logits -> probabilities
            for (int el = lane; el < npairs; el += WAVE)
                C.prob[(size_t)(e0 + el) * H + h] = hw_exp2((logit_s[el] - m_run) * LOG2E) * inv;
        } else {
            for (int g0 = 0; g0 < npairs; g0 += FC_GROUP) {      // each was written by the lane that now reads it
                if (sub == 0 && g0 + pr < npairs) {
                    const size_t eh = (size_t)(e0 + g0 + pr) * H + h;
                    C.prob[eh] = hw_exp2((C.prob[eh] - m_run) * LOG2E) * inv;
                }
            }
        }
        if (PLACES && !own && it_cur < C.ticket_items) core_project_done<HWK>(C, it_cur, h, lane);
        count_item();
    }
}

// The product of four channels (from c0 on) of a handed-over item with the weights, which wait in registers: the same sums as the
// item's own wavefront makes.
template <int HWK>
struct CoreProductWeights {
    static constexpr bool VEC = HWK >= 4 * WAVE;
    static constexpr int NW = VEC ? (HWK / 4 + WAVE - 1) / WAVE : 1, NV = VEC ? 4 * NW : HWK / WAVE;
    float w[4][NV];
    __device__ __forceinline__ void load(const float* __restrict__ wcat, int h, int c0, int lane) {
        const float* Wh = wcat + ((size_t)h * DH + c0) * HWK;
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int u = 0; u < (VEC ? NW : NV); u++) {
                if (VEC) {      // (a lane past the end reads the last words; its own are zero)
                    const float4 t = *reinterpret_cast<const float4*>(Wh + c * HWK + 4 * min(lane + WAVE * u, HWK / 4 - 1));
                    w[c][4 * u] = t.x; w[c][(4 * u + 1) % NV] = t.y; w[c][(4 * u + 2) % NV] = t.z; w[c][(4 * u + 3) % NV] = t.w;
                } else {
                    w[c][u] = Wh[c * HWK + lane + WAVE * u];
                }
            }
    }
    __device__ __forceinline__ void product(const int32_t* hist, const float4* tab, float* out, int h, int H, int c0, int lane) const {
        float word[NV], v[4];
#pragma unroll
        for (int u = 0; u < (VEC ? NW : NV); u++) {
            if (VEC) {
                int4 t = make_int4(0, 0, 0, 0);
                if (lane + WAVE * u < HWK / 4) t = reinterpret_cast<const int4*>(hist)[lane + WAVE * u];
                word[4 * u] = __int_as_float(t.x); word[(4 * u + 1) % NV] = __int_as_float(t.y);
                word[(4 * u + 2) % NV] = __int_as_float(t.z); word[(4 * u + 3) % NV] = __int_as_float(t.w);
            } else {
                word[u] = __int_as_float(hist[lane + WAVE * u]);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            v[c] = lane == ((c0 + c) >> 1) ? reinterpret_cast<const float*>(tab)[c0 + c] : 0.0f;
#pragma unroll
            for (int u = 0; u < (VEC ? NW : NV); u++)
                v[c] = VEC ? fmaf(word[4 * u], w[c][4 * u], fmaf(word[(4 * u + 1) % NV], w[c][(4 * u + 1) % NV],
                             fmaf(word[(4 * u + 2) % NV], w[c][(4 * u + 2) % NV], fmaf(word[(4 * u + 3) % NV], w[c][(4 * u + 3) % NV], v[c]))))
                           : fmaf(word[u], w[c][u], v[c]);
        }
        const float sum = wave_sum4(v, lane);
        const int i = __float_as_int(tab[4].x);
        if ((lane & 15) == 0) out[((size_t)i * H + h) * DH + c0 + (lane >> 4)] = sum;
    }
};

// ---- inference without the angle encoding: several heads of an atom in one wavefront ------------------------------
// Without frames nothing but a, q, k and v differs from head to head: the pairs' vectors and distances, the walk over the sorted
// table, the list of the images and the ratios of the distance window are made once for HEADS items, the lanes of a row of eight
// share out the heads for what is made once per (pair, head).  For items with the usual box, whose nearest images are known.
// The kernel of one item per wavefront was bound by vector-instruction issue (138 M instructions for 180 224 items; four heads 69 M);
// what bounds this one are LDS atomics and vector instructions alike (67 and 53 % with one copy of the bins).  4096 crystals,
// four layers: 1306 us -> 1000.  With the angle encoding (built for 64 and 16 bins, two and four heads: 26 and 38 % fewer vector
// instructions) the histograms leave room for too few wavefronts: 2650 -> 2654, 2830 us; training 1320 -> 1336, 1403.
template <int HEADS>
struct CoreHeadsShared {
    using Hist = CoreHist<0, true, 4>;
    struct Pair { float4 A; float C[HEADS]; };      // rx, ry, rz, d2min; per head exp(logit - running max) / S in fixed-point units
    float4 tab[FC_TCAP];
    uint16_t list[FC_LISTCAP];
    __attribute__((aligned(16))) int32_t hist[HEADS][Hist::ALL];
    __attribute__((aligned(16))) Pair pair[FC_GROUP];
};
__device__ __forceinline__ float rows8_max(float x) {
    x = fmaxf(x, dpp_move<0x128>(x));          // row_ror 8: the other half of the 16-lane row
    return -rows_min(-x);
}
// The records of HEADS heads of an item: words of heads 2 k, 2 k + 1 in the two halves of rec[k].
template <int HEADS>
struct HeadRecords {
    uint32_t rec[HEADS / 2];
    __device__ __forceinline__ void load(const KernelArgs& P, int it, int h0, int lane) {
#pragma unroll
        for (int k = 0; k < HEADS / 2; k++) rec[k] = P.items[((size_t)it * P.H + h0 + 2 * k) * REC_WORDS + lane];
    }
    __device__ __forceinline__ int word(int head, int w) const { return __builtin_amdgcn_readlane((int)rec[head >> 1], (head & 1) * REC_WORDS + w); }
};
template <int WL, int HEADS>
__device__ __forceinline__ void fused_core_fwd_heads(const CoreArgs& C, CoreHeadsShared<HEADS>& sh, int h0, const HeadRecords<HEADS>& rec) {
    static_assert(WL > 0 && (HEADS == 2 || HEADS == 4), "");
    using Hist = typename CoreHeadsShared<HEADS>::Hist;
    constexpr int LPH = FC_GROUP / HEADS;      // lanes of a row per head
    constexpr int CH4 = HEADS / 2;             // 16-byte pieces of a head's 16 channels per lane
    float4* const tab = sh.tab;
    uint16_t* const list = sh.list;
    const KernelArgs& P = C.K;
    const BasisConsts bc = P.bc;
    const int lane = threadIdx.x & (WAVE - 1), pr = lane >> 3, sub = lane & 7, H = P.H;
    const int hs = sub / LPH, ck = sub % LPH;      // this lane's head and its part of the head's channels
    const float prune = (P.prune_log2 > 0.0f) ? -P.prune_log2 : -3.0e38f;
    const float INF = __builtin_inff();
    const int i = rec.word(0, REC_ATOM), e0 = rec.word(0, REC_E0), npairs = rec.word(0, REC_NPAIRS), j0 = rec.word(0, REC_J0);
    const int crystal = rec.word(0, REC_CRYSTAL);
    const int s0 = 2 * C.table_R + 1, T = s0 * s0 * s0;
    // operands of the pair served by this row, fetched one group ahead
    float nrx = 0.f, nry = 0.f, nrz = 0.f, nnear = 0.f;
    float4 nk[CH4], nv[CH4], q4[CH4];
    auto fetch = [&](int g0) {
        // (no branch per row: a row past the end re-reads the row's last pair; nothing of it is used)
        const uint32_t el = (uint32_t)min(g0 + pr, npairs - 1);
        const uint32_t e = min((uint32_t)e0 + el, (uint32_t)(P.E - 1));
        const uint32_t jh = ((((uint32_t)j0 + el) * (uint32_t)H + (uint32_t)(h0 + hs)) * DH + 4u * CH4 * ck) * 4u;
        const float3 r3 = load_at<float3>(P.rpos, e * 12u);
        nrx = r3.x; nry = r3.y; nrz = r3.z;
#pragma unroll
        for (int c = 0; c < CH4; c++) { nk[c] = load_at<float4>(C.k, jh + 16u * c); nv[c] = load_at<float4>(C.v, jh + 16u * c); }
        nnear = load_at<float>(C.pair_near, e * 8u);
    };
    float4 acc[CH4];                           // sum_j exp(logit_j - m_run) v_j of this lane's channels
    {
        const float4* src = C.sorted_tab + (size_t)crystal * FC_TCAP;
        const float4 ta = src[lane], tb = src[lane + WAVE];
        const uint32_t qo = (((uint32_t)i * (uint32_t)H + (uint32_t)(h0 + hs)) * DH + 4u * CH4 * ck) * 4u;
#pragma unroll
        for (int c = 0; c < CH4; c++) {
            q4[c] = load_at<float4>(C.qs, qo + 16u * c);
            acc[c] = nk[c] = nv[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (npairs > 0) fetch(0);
#pragma unroll
        for (int hh = 0; hh < HEADS; hh++) Hist::clear(sh.hist[hh], lane);
        tab[lane] = ta;
        tab[lane + WAVE] = tb;
    }
    float a2[HEADS], a_own = 0.0f, a2_far = -INF;      // a2_far: of the head that sees farthest
#pragma unroll
    for (int hh = 0; hh < HEADS; hh++) {
        const float a = __int_as_float(rec.word(hh, REC_A));
        a2[hh] = a * LOG2E;
        a2_far = fmaxf(a2_far, a2[hh]);
        a_own = hs == hh ? a : a_own;
    }
    const float cutS = C.skip_log2 * hw_rcp(-a2_far);      // (a bound with margins)
    const int dist0 = Hist::dist_word(lane);
    const float fixs = 1073741824.0f * hw_rcp((float)max(npairs, 1));      // (see fused_core_fwd_body)
    float m_run = -INF, Dl = 0.0f;             // running maximum of the logits, share of the denominator: of this lane's head
    unsigned long long n_eval = 0, n_seen = 0;
    const bool count = P.stats != nullptr;
    wave_sync();

    for (int g0 = 0; g0 < npairs; g0 += FC_GROUP) {
        const float rx = nrx, ry = nry, rz = nrz, d2min = nnear;
        float4 k4[CH4], v4[CH4];
#pragma unroll
        for (int c = 0; c < CH4; c++) { k4[c] = nk[c]; v4[c] = nv[c]; }
        if (g0 + FC_GROUP < npairs) fetch(g0 + FC_GROUP);
        const bool active = g0 + pr < npairs;
        // ---- one walk over the table: weights, normalisers, the images that any head keeps
        const float rn = hw_sqrt(fmaf(rx, rx, fmaf(ry, ry, rz * rz)));
        const float reach = fmaf(1.0001f, rn + hw_sqrt(d2min + cutS), 1e-4f);
        const float lim = active ? fminf(reach, FC_REACH_ALL) : -1.0f;      // (lengths are >= 0; padding: +inf)
        float Sb[HEADS];
#pragma unroll
        for (int hh = 0; hh < HEADS; hh++) Sb[hh] = 0.0f;
        int nlist = 0;
        {
            float4 v = tab[sub];
            for (int t0 = 0; t0 < T; t0 += FC_GROUP) {
                const int t = t0 + sub;
                const float4 vn = tab[min(t + FC_GROUP, FC_TCAP - 1)];      // the next step's entry, in flight meanwhile
                const bool in = v.w <= lim;
                const uint64_t inm = ballot(in);
                if (inm == 0) break;                             // every row is past its reach (lengths ascend)
                const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
                const float de = in ? fmaf(dx, dx, fmaf(dy, dy, dz * dz)) - d2min : INF;      // (a < 0: weight 2^-inf = 0)
                bool keep = false;
#pragma unroll
                for (int hh = 0; hh < HEADS; hh++) {
                    const float ex = a2[hh] * de;
                    Sb[hh] += hw_exp2(ex);
                    keep = keep || ex >= prune;
                    if (count) n_eval += __popcll(ballot(ex >= prune));
                }
                n_seen += (unsigned long long)(HEADS * __popcll(inm));
                const uint64_t m = ballot(keep);
                if (keep) list[nlist + lane_prefix(m)] = (uint16_t)((pr << FC_SHIFT) | t);
                nlist += __popcll(m);
                v = vn;
            }
        }
        // ---- logits, running softmax: a lane per (pair, head, part of the channels)
        float S = 0.0f;
#pragma unroll
        for (int hh = 0; hh < HEADS; hh++) { const float Sh = half_sum(Sb[hh]); S = hs == hh ? Sh : S; }
        float qk = 0.0f;
#pragma unroll
        for (int c = 0; c < CH4; c++)
            qk += fmaf(q4[c].x, k4[c].x, q4[c].y * k4[c].y) + fmaf(q4[c].z, k4[c].z, q4[c].w * k4[c].w);
        qk += dpp_move<0xB1>(qk);
        if (LPH == 4) qk += dpp_move<0x4E>(qk);
        const float z = fmaf(hw_log2(S), LN2, a_own * d2min);
        const float logit = active ? qk + z : -INF;
        const float gmax = rows8_max(logit);
        const bool grow = gmax > m_run;
        const uint64_t rescaled = ballot(grow && m_run > -INF);
        if (rescaled) {
            const float fac = grow && m_run > -INF ? hw_exp2((m_run - gmax) * LOG2E) : 1.0f;
#pragma unroll 1
            for (int hh = 0; hh < HEADS; hh++)
                if ((rescaled >> (hh * LPH)) & 1)
                    Hist::rescale(sh.hist[hh], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fac), hh * LPH)), lane);
#pragma unroll
            for (int c = 0; c < CH4; c++) { acc[c].x *= fac; acc[c].y *= fac; acc[c].z *= fac; acc[c].w *= fac; }
            Dl *= fac;
        }
        m_run = grow ? gmax : m_run;
        const float ew = active ? hw_exp2((logit - m_run) * LOG2E) : 0.0f;
#pragma unroll
        for (int c = 0; c < CH4; c++) {
            acc[c].x = fmaf(ew, v4[c].x, acc[c].x); acc[c].y = fmaf(ew, v4[c].y, acc[c].y);
            acc[c].z = fmaf(ew, v4[c].z, acc[c].z); acc[c].w = fmaf(ew, v4[c].w, acc[c].w);
        }
        Dl += ew;
        if (sub == 0 && active) sh.pair[pr].A = make_float4(rx, ry, rz, d2min);
        if (ck == 0 && active) sh.pair[pr].C[hs] = ew * hw_rcp(S) * fixs;
        wave_sync();
        // ---- the images of the list, into every head's histogram (an image that only others keep is left out)
        for (int base = 0; base < nlist; base += WAVE) {
            const int idx = base + lane;
            if (idx < nlist) {
                const uint32_t ent = list[idx];
                const float4 v = tab[ent & (FC_TCAP - 1)];
                const auto& pp = sh.pair[ent >> FC_SHIFT];
                const float4 pa = pp.A;
                float pc[HEADS];
#pragma unroll
                for (int hh = 0; hh < HEADS; hh++) pc[hh] = pp.C[hh];
                const float dx = pa.x + v.x, dy = pa.y + v.y, dz = pa.z + v.z;
                const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                const float de = d2 - pa.w;
                const float u = hw_sqrt(d2) * bc.inv_interval;
                int start = (int)(u - bc.start_off);          // truncation toward zero
                start = max(0, min(start, NBINS - WL));
                const float beta_c = ((float)(start + WL / 2 + 1) - u) * bc.len_step;
                const WindowSeed s = window_seed(beta_c, bc.len_step, 1.0f);
                float rr[WL / 2], rl[WL / 2];                 // from bin to bin outwards from the window's centre
                rr[0] = s.rr; rl[0] = s.rl;
#pragma unroll
                for (int m = 1; m < WL / 2; m++) { rr[m] = rr[m - 1] * bc.len_cc; rl[m] = rl[m - 1] * bc.len_cc; }
                start += dist0;
#pragma unroll
                for (int hh = 0; hh < HEADS; hh++) {
                    const float ex = a2[hh] * de;
                    if (ex >= prune) {
                        const float gc = s.gc * (hw_exp2(ex) * pc[hh]);
                        int32_t* const hb = sh.hist[hh] + start;
                        atomicAdd(hb + WL / 2, rint_i(gc));
                        float g = gc;
#pragma unroll
                        for (int m = 0; m < WL / 2; m++) { g *= rr[m]; atomicAdd(hb + WL / 2 + 1 + m, rint_i(g)); }
                        g = gc;
#pragma unroll
                        for (int m = 0; m < WL / 2; m++) { g *= rl[m]; atomicAdd(hb + WL / 2 - 1 - m, rint_i(g)); }
                    }
                }
            }
        }
        wave_sync();                      // list and pair data may be rewritten
    }

    // ---- the rows are complete: normalise and write
    const float D = rows8_sum(Dl);
    const float inv = D > 0.0f ? hw_rcp(D) : 0.0f;
    const float sc_own = inv * hw_rcp(fixs);
    {
        float* const dst = C.out + ((size_t)i * H + h0) * DH;      // (the heads' channels are contiguous)
#pragma unroll
        for (int c = 0; c < CH4; c++) {
            const float4 o = make_float4(rows8_sum(acc[c].x) * inv, rows8_sum(acc[c].y) * inv, rows8_sum(acc[c].z) * inv, rows8_sum(acc[c].w) * inv);
            if (lane < FC_GROUP) reinterpret_cast<float4*>(dst)[sub * CH4 + c] = o;
        }
    }
#pragma unroll
    for (int hh = 0; hh < HEADS; hh++) {
        const float sc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc_own), hh * LPH));
        static_assert(HW_DIST == WAVE, "a word per lane");
        C.hist[((size_t)(h0 + hh) * P.N + i) * HW_DIST + lane] = (float)Hist::word(sh.hist[hh], lane) * sc;
    }
    if (count && lane == 0) {
        atomicAdd(P.stats + STAT_FWD_EVAL, n_eval);
        atomicAdd(P.stats + STAT_FWD_RAW, (unsigned long long)HEADS * (unsigned long long)T * (unsigned long long)npairs);
        atomicAdd(P.stats + STAT_FWD_PAIRS, (unsigned long long)HEADS * (unsigned long long)npairs);
        atomicAdd(P.stats + STAT_FWD_SEEN, n_seen);
    }
}
// The leading wavefronts take a listed record each, the next ones HEADS heads of an atom (where some of those are listed, the others
// one after the other), and the `rest` last ones, as many as are resident, the listed records that are left: the first by their own
// rank, the next ones as they come from NQUEUE counters, until there are no more (they wait at the list for what they take next,
// where a wavefront per item waits for its turn at the dispatcher).
// Records with a box of their own have 18 wavefronts per compute unit here (LDS) and 28 in the kernel of one item per wavefront.
// Whole passes of four layers in us, that kernel / this one: nothing but such cells, 22 000 items 999/1004, 66 000 items 2601/2655
// (dealt out beforehand and looked up in the lists twice, at 16 per compute unit: 3111); half of them so 1611/1576; one in ten 851/766;
// ordinary cells, 180 224 items, 1305/960.  Five wavefronts per SIMD with four heads: 96 registers instead of 103, 1036 -> 1017 for the
// ordinary cells of another machine.  Two records per draw: 22 000 items 1005 -> 1059.
template <int WL, int HEADS>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(HEADS == 4 ? 5 : 1)))
void fused_core_fwd_heads_kernel(const CoreArgs C, int rest) {
    __shared__ union { CoreFwdLds<0, true> one; CoreHeadsShared<HEADS> several; } sh;
    const KernelArgs& P = C.K;
    const int lane = (int)threadIdx.x & (WAVE - 1), w = (int)blockIdx.x;
    const int groups = P.N * P.H / HEADS;
    const bool by_rank = w < C.slow_wgs || w >= C.slow_wgs + groups;
    int wid = 0, rank = w < C.slow_wgs ? w : w - groups;
    uint32_t left = 0;                 // heads of this wavefront's own that are not listed
    if (!by_rank) {
        constexpr int shift = HEADS == 2 ? CORE_DIE_SHIFT - 1 : CORE_DIE_SHIFT - 2;      // (an atom's heads on one die)
        wid = HEADS * __builtin_amdgcn_readfirstlane(die_order(w - C.slow_wgs, groups, shift));
        const int it = div_heads(P, wid), h0 = wid - it * P.H;
        if (it >= P.N) return;
        HeadRecords<HEADS> rec;
        rec.load(P, it, h0, lane);
        const int usual = C.table_R | (C.table_R << 8) | (C.table_R << 16);
        bool together = true;
#pragma unroll
        for (int hh = 0; hh < HEADS; hh++) {
            const int box = rec.word(hh, REC_BOX);
            together = together && box == usual && __int_as_float(rec.word(hh, REC_A)) < 0.0f;
            left |= ((uint32_t)box & REC_BOX_LISTED) != 0u ? 0u : 1u << hh;
        }
        if (together) {
            fused_core_fwd_heads<WL, HEADS>(C, sh.several, h0, rec);
            return;
        }
    }
    SlowRuns runs{0, 0};
    if (by_rank) runs = core_slow_runs(C, lane);
#pragma unroll 1
    for (;;) {
        int item;
        if (by_rank) {
            item = __builtin_amdgcn_readfirstlane(core_slow_record(C, runs, rank, lane));
            if (item < 0) return;
        } else {
            if (left == 0) return;
            item = wid + __builtin_ctz(left);
            left &= left - 1;
        }
        wave_sync();
        fused_core_fwd_body<WL, 0, false, true>(C, sh.one, item, nullptr, nullptr, true);
        if (w < C.slow_wgs) return;
        if (by_rank) {
            const int q = w & (NQUEUE - 1);
            rank = C.slow_wgs + rest + queue_draw(P.counters + q * QSTRIDE) * NQUEUE + q;
        }
    }
}

// (distance encoding alone: 4.8 KB of LDS per item allow eight wavefronts per SIMD; seven, with 72 registers and
// nothing spilled, ran faster than eight with 64 and nine spilled)
template <int WL, int ANG, bool COS_ABS, bool LEAN = false>
__global__ __launch_bounds__(WAVE * CORE_WPB) __attribute__((amdgpu_waves_per_eu(ANG > 0 ? 1 : 7)))
void fused_core_fwd_kernel(const CoreArgs C) {
    constexpr int COPIES = LEAN && ANG == NBINS ? 2 : 1;
    __shared__ CoreFwdLds<ANG, LEAN, COPIES> shared[CORE_WPB];
    const int wid = core_wave_record(C, (int)blockIdx.x * CORE_WPB + (int)(threadIdx.x >> 6), (int)threadIdx.x & (WAVE - 1));
    if (wid >= 0) fused_core_fwd_body<WL, ANG, COS_ABS, LEAN, COPIES>(C, shared[threadIdx.x >> 6], wid);
}

// A workgroup per sixteen items and head, a wavefront per slice; the slices meet in LDS and the first wavefront adds them in
// their order.  PLACES: histograms in the order of the sixteens, from sixteen `first` on; else in the order of the atoms,
// sixteen consecutive ones.  grid (sixteens, H).
template <int HWK, bool PLACES>
__global__ __launch_bounds__(WAVE * ProjectSlices<HWK>::N) void core_project_kernel(const float* __restrict__ hist,
        const float* __restrict__ wcat, const uint32_t* __restrict__ records, float* __restrict__ out, int N, int H, int first) {
    using S = ProjectSlices<HWK>;
    __shared__ float part[S::N][4][WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x >> 6, col = lane & 15, kk = lane >> 4;
    const int h = blockIdx.y, sixteen = first + (int)blockIdx.x;
    const int members = PLACES ? sixteen_members(sixteen, N) : min(16, N - sixteen * 16);
    if (members <= 0) return;
    ProjectRow R;
    if (PLACES) R = project_row(records, sixteen, members, h, H, lane);
    else R.row = R.atom = min(sixteen * 16 + col, N - 1);
    const float4* ap = reinterpret_cast<const float4*>(hist + ((size_t)h * (PLACES ? project_rows(N) : N) + R.row) * HWK +
                                                       wv * S::UNITS * 16) + kk;
    const float4* bp = reinterpret_cast<const float4*>(wcat + ((size_t)h * DH + col) * HWK + wv * S::UNITS * 16) + kk;
    const v4f_c acc = project_slice<S::UNITS, S::UNITS>([&](int u) { return ap[4 * u]; }, bp);
#pragma unroll
    for (int r = 0; r < 4; r++) part[wv][r][lane] = acc[r];
    __syncthreads();
    if (wv != 0) return;
    // component r of lane (kk, col): rank 4 kk + r, channel col
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float sum = part[0][r][lane];
#pragma unroll
        for (int w = 1; w < S::N; w++) sum += part[w][r][lane];
        const int i = PLACES ? __shfl(R.atom, 4 * kk + r) : sixteen * 16 + 4 * kk + r;
        if (4 * kk + r < members) out[((size_t)i * H + h) * DH + col] += sum;
    }
}

// G (H,N,hw) = go (N,H,16) . Wcat_h (16, hw): wavefront per (16 atoms, head, 64-word block); four MFMA tiles whose
// columns are interleaved (tile t, column c <-> word 4 c + t) so that a lane stores 16 consecutive bytes.
// grid (ceil(N/16), H, hw/64).  `queues`: optional work-queue heads to clear (when no prepare launch does).
// Records kept from the forward pass (`slow.items` not null): the wavefronts (x, 0, 0) with x a multiple of
// SLOW_GB_BLOCKS also list the records of SLOW_GB_BLOCKS x 16 atoms whose box is not the usual one, for the main kernel of the backward pass to take first (as prepare_items_block does for the forward,
// whose lists are gone by now).
constexpr int SLOW_GB_BLOCKS = 4;
struct SlowListArgs {
    uint32_t* items;       // (N, H, REC_WORDS) or null
    int32_t* count;        // (lists), lists = ceil(ceil(N / 16) / SLOW_GB_BLOCKS)
    int32_t* list;         // (lists, SLOW_GB_BLOCKS x 16 x H)
    int32_t R;             // half-width of the usual box
};
__global__ __launch_bounds__(WAVE) void core_gbuild_kernel(const float* __restrict__ go, const float* __restrict__ wcat,
                                                           float* __restrict__ G, int N, int H, int hw,
                                                           int32_t* __restrict__ queues, const SlowListArgs slow) {
    const int lane = threadIdx.x, col = lane & 15, kk = lane >> 4;
    const int h = blockIdx.y, i0 = blockIdx.x * 16;
    if (queues && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0)      // work queues of the launch that follows
        for (int u = lane; u < H * NQUEUE; u += WAVE) queues[u * QSTRIDE] = 0;
    if (slow.items && blockIdx.y == 0 && blockIdx.z == 0 && blockIdx.x % SLOW_GB_BLOCKS == 0) {
        const int li = (int)blockIdx.x / SLOW_GB_BLOCKS;
        const int first = (int)blockIdx.x * 16 * H, last = min(first + SLOW_GB_BLOCKS * 16 * H, N * H);
        const uint32_t usual = (uint32_t)(slow.R | (slow.R << 8) | (slow.R << 16));
        int listed = 0;
        for (int r0 = first; r0 < last; r0 += 4 * WAVE) {
            // (four loads that do not wait for each other, then their ranks)
            uint32_t boxw[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int r = r0 + u * WAVE + lane;
                boxw[u] = r < last ? slow.items[(size_t)r * REC_WORDS + REC_BOX] : usual;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int r = r0 + u * WAVE + lane;
                const bool own = r < last && (boxw[u] & 0x00ffffffu) != usual;
                const uint64_t m = ballot(own);
                const int rank = listed + __popcll(m & ((1ull << lane) - 1ull));
                if (r < last) {
                    if (own) slow.list[(size_t)li * (SLOW_GB_BLOCKS * 16 * H) + rank] = r;
                    const uint32_t neww = own ? (boxw[u] | REC_BOX_LISTED_BWD) : (boxw[u] & ~REC_BOX_LISTED_BWD);
                    if (neww != boxw[u]) slow.items[(size_t)r * REC_WORDS + REC_BOX] = neww;
                }
                listed += __popcll(m);
            }
        }
        if (lane == 0) slow.count[li] = listed;
    }
    const int row = min(i0 + col, N - 1);
    const float4 a4 = reinterpret_cast<const float4*>(go + ((size_t)row * H + h) * DH)[kk];      // channels 4 kk ..
    const float A[4] = {a4.x, a4.y, a4.z, a4.w};
    {
        const int w0 = blockIdx.z * 64;
        float4 b4[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            b4[j] = *reinterpret_cast<const float4*>(wcat + ((size_t)h * DH + 4 * kk + j) * hw + w0 + 4 * col);
        v4f_c acc[4];
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = v4f_c{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j], b4[j].x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j], b4[j].y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j], b4[j].z, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j], b4[j].w, acc[3], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int it = i0 + 4 * kk + r;
            if (it < N)
                *reinterpret_cast<float4*>(G + ((size_t)h * N + it) * hw + w0 + 4 * col) =
                    make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]);
        }
    }
}

// gwcat (slice,H,16,hw) = sum over a slice of the atoms of go (.,h,16) (x) hist (h,.,hw): wavefront per (head, 64-word
// block, slice); four MFMA tiles with interleaved columns as above.  grid (ceil(hw/64 / GW_WPB), H, nslices), at most
// CORE_GW_SLICES slices.
__device__ __forceinline__ void core_gwcat_block(const float* __restrict__ go, const float* __restrict__ hist,
                                                 float* __restrict__ gwcat, int N, int H, int hw, int per_slice, int slice) {
    // the GW_WPB wavefronts of a workgroup take neighbouring pieces of the same rows at the same time: GW_WPB x 256
    // contiguous bytes of a row instead of 256 bytes every 4 KB (82 -> 70 us for the four layers of the benchmark)
    const int lane = threadIdx.x & (WAVE - 1), col = lane & 15, kk = lane >> 4;
    const int w0 = ((int)blockIdx.x * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6)) * 64, h = blockIdx.y;
    if (w0 >= hw) return;
    const int i_begin = slice * per_slice, i_end = min(N, i_begin + per_slice);
    v4f_c acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) acc[t] = v4f_c{0.f, 0.f, 0.f, 0.f};
    // GW_DEPTH x 16 atoms per step, all their loads asked for before the first product: a wavefront keeps 16 KB of
    // histogram rows in flight (with 4 KB the kernel ran at 40 % of the bandwidth it reaches now)
    constexpr int GW_DEPTH = 4;
    for (int ib = i_begin; ib < i_end; ib += 16 * GW_DEPTH) {
        float av[GW_DEPTH][4];
        float4 bv[GW_DEPTH][4];
#pragma unroll
        for (int d = 0; d < GW_DEPTH; d++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // (no branch around the loads: an atom past the end reads the slice's first one, with go as zero)
                const int it = ib + 16 * d + 4 * j + kk;
                const bool live = it < i_end;
                const int itc = live ? it : i_begin;
                const float g = go[((size_t)itc * H + h) * DH + col];
                av[d][j] = live ? g : 0.0f;
                bv[d][j] = *reinterpret_cast<const float4*>(hist + ((size_t)h * N + itc) * hw + w0 + 4 * col);
            }
        // (without the branches the compiler would put every load next to its product: 113 us instead of 78)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < GW_DEPTH; d++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][j], bv[d][j].x, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][j], bv[d][j].y, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][j], bv[d][j].z, acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][j], bv[d][j].w, acc[3], 0, 0, 0);
            }
    }
    // component r of tile t, lane (kk, col): channel 4 kk + r, word w0 + 4 col + t.  Every slice writes its own
    // copy (slice, H, 16, hw) in full: nothing to clear, no atomics, and the sum over the slices that follows is made
    // in a fixed order
    float* const part = gwcat + (size_t)slice * H * DH * hw;
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<float4*>(part + ((size_t)h * DH + 4 * kk + r) * hw + w0 + 4 * col) =
            make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]);
}
constexpr int GW_WPB = 4;          // wavefronts per workgroup of the two kernels below (8: the same; 16: far slower)
__global__ __launch_bounds__(WAVE * GW_WPB) void core_gwcat_kernel(const float* __restrict__ go, const float* __restrict__ hist,
                                                          float* __restrict__ gwcat, int N, int H, int hw, int per_slice) {
    core_gwcat_block(go, hist, gwcat, N, H, hw, per_slice, (int)blockIdx.z);
}
// several jobs: grid (ceil(hw/64 / GW_WPB), H, slices of all jobs); the job of a slice by a scan of the (few) jobs
__global__ __launch_bounds__(WAVE * GW_WPB) void core_gwcat_multi_kernel(const CoreWgradJobs T) {
    int j = 0;
    while (j + 1 < T.njobs && (int)blockIdx.z >= T.job[j + 1].slice0) j++;
    const CoreWgradJob& J = T.job[j];
    core_gwcat_block(J.go, J.hist, J.gwcat, J.N, T.H, T.hw, J.per_slice, (int)blockIdx.z - J.slice0);
}
// grid (H*16, jobs): added to the destinations (or written)
__global__ __launch_bounds__(256) void core_gw_finish_multi_kernel(const CoreWgradJobs T) {
    const CoreWgradJob& J = T.job[blockIdx.y];
    core_gw_finish_block(J.gwcat, J.nslices, (size_t)T.H * DH * T.hw, T.hw, T.dist_coef, T.angle_coef, T.ws,
                         J.gW[0], J.gW[1], J.gW[2], J.gW[3], (int)blockIdx.x, T.overwrite == 0);
}


// =================================================================================================================
// backward
// =================================================================================================================
// Per item: G = Wcat^T go (made by core_gbuild_kernel) in LDS; for every image n of pair j with probability
// p_n = exp(a d^2 - z) the value bg_n = sum_k b_k(d_n) G_k + sum_axis sum_o eps^o G'_(axis,o,m*) is gathered, and
//     go . psi_ij          = sum_n p_n bg_n                                   (per pair, fixed-point LDS sums)
//     gl_ij = dL/dlogit_ij = P_ij (go . v_j + go . psi_ij - go . out_i)
//     ga_ih                = sum_j P_ij [(go . v_j - go . out_i) A0_j + sum_n p_n d_n^2 bg_n],  A0_j = sum_n p_n d_n^2
//     gq_i                 = sum_j gl_ij k_j
// (the terms A0_j (go . psi_ij) of dL/dz and of the covariance form cancel).  gk and gv are sums over the pairs that
// point AT an atom and are left to the column kernel of the attention backward (from gl and P).
template <int HWK>
struct CoreBwdShared {
    float4 tab[FC_TCAP];
    uint16_t list[FC_LISTCAP];
    float Gs[HWK];
    float4 pairA[FC_GROUP];      // rx, ry, rz, z log2(e)
    float pairP[FC_GROUP];       // P_ij
    int32_t pairB[FC_GROUP];     // sum_n P_ij p_n bg_n in fixed point
};
template <int WL, int ANG, bool COS_ABS>
__global__ __launch_bounds__(WAVE * CORE_WPB) void fused_core_bwd_kernel(const CoreArgs C) {
    constexpr bool HAS_ANG = ANG > 0;
    constexpr int HWK = core_hist_words(ANG);
    __shared__ CoreBwdShared<HWK> shared[CORE_WPB];
    CoreBwdShared<HWK>& sh = shared[threadIdx.x >> 6];
    float4* const tab = sh.tab;
    uint16_t* const list = sh.list;
    float* const Gs = sh.Gs;
    float4* const pairA = sh.pairA;
    float* const pairP = sh.pairP;
    int32_t* const pairB = sh.pairB;

    const KernelArgs& P = C.K;
    const int lane = threadIdx.x & (WAVE - 1);
    const int H = P.H;
    const int wid = core_wave_record(C, (int)blockIdx.x * CORE_WPB + (int)(threadIdx.x >> 6), lane);
    if (wid < 0) return;
    const int it_cur = div_heads(P, wid);      // one wavefront per item, long items first
    const int h = wid - it_cur * H;
    const int pr = lane >> 3, sub = lane & 7;
    const BasisConsts bc = P.bc;
    const int WLr = WL > 0 ? WL : bc.len_window;      // bins of the distance window (WL == 0: known at run time only)
    const float prune = (P.prune_log2 > 0.0f) ? -P.prune_log2 : -3.0e38f;
    const float INF = __builtin_inff();

    if (it_cur >= P.N) return;
    {
        const uint32_t rec_cur = load_record_lane(P, it_cur, h, lane);
        if (core_record_taken_elsewhere(C, rec_cur, wid, lane)) return;
        const CoreItem ci = core_unpack(C, rec_cur, true);
        const int i = ci.item.i;
        const float a2 = ci.item.a * LOG2E;
        const Lattice L = ci.item.L;
        const Box bx = ci.item.bx;
        const bool sorted = ci.sorted;
        const int nchunks = ci.nchunks;
        float f[3][3];
        if (HAS_ANG) {
#pragma unroll
            for (int ax = 0; ax < 3; ax++)
#pragma unroll
                for (int d = 0; d < 3; d++) f[ax][d] = rec_f(rec_cur, REC_FRAMES + ax * 3 + d);
        }
        const int e0 = ci.item.e0, npairs = ci.item.npairs;
        const size_t ih = (size_t)i * H + h;
        core_load_table(C, ci, tab, lane);
        float gabs = 0.0f;
        {
            const float* src = C.G + ((size_t)h * P.N + i) * HWK;
            if (HWK >= 4 * WAVE) {
                constexpr int NW = HWK >= 4 * WAVE ? HWK / (4 * WAVE) : 1;
                float4 g4[NW];
#pragma unroll
                for (int u = 0; u < NW; u++) g4[u] = reinterpret_cast<const float4*>(src)[lane + WAVE * u];
#pragma unroll
                for (int u = 0; u < NW; u++) {
                    reinterpret_cast<float4*>(Gs)[lane + WAVE * u] = g4[u];
                    gabs += (fabsf(g4[u].x) + fabsf(g4[u].y)) + (fabsf(g4[u].z) + fabsf(g4[u].w));
                }
            } else {
                for (int u = lane; u < HWK; u += WAVE) { const float g = src[u]; Gs[u] = g; gabs += fabsf(g); }
            }
        }
        const float2 go2 = *reinterpret_cast<const float2*>(C.go + ih * DH + 2 * sub);
        const float2 ov2 = *reinterpret_cast<const float2*>(C.outv + ih * DH + 2 * sub);
        const float c0 = half_sum(fmaf(go2.x, ov2.x, go2.y * ov2.y));          // go . out_i
        const float gnorm = uniform_f(wave_sum(gabs));                          // |bg| <= sum |G|
        const float inv_a2 = a2 < 0.0f ? hw_rcp(a2) : 0.0f;             // (for a bound with margins)
        const float bscale = 1073741824.0f / fmaxf(gnorm, 1e-20f);      // (finite: 2^30 / 1e-30 would not be)
        const float binv = fmaxf(gnorm, 1e-20f) * (1.0f / 1073741824.0f);
        wave_sync();
        float cov = 0.0f;
        float2 gq2 = make_float2(0.f, 0.f);
        unsigned long long n_eval = 0;

        float nrx = 0.f, nry = 0.f, nrz = 0.f, nz = 0.f, npb = 0.f;
        float2 nk2 = make_float2(0.f, 0.f), nv2 = nk2;
        auto fetch = [&](int g0) {
            // (no branch per row: a row past the end re-reads the row's last pair; nothing of it is used)
            const uint32_t el = (uint32_t)min(g0 + pr, npairs - 1);
            const uint32_t e = min((uint32_t)e0 + el, (uint32_t)(P.E - 1));
            const uint32_t jh = ((((uint32_t)ci.j0 + el) * (uint32_t)H + (uint32_t)h) * DH + 2u * sub) * 4u;
            const uint32_t eh = (e * (uint32_t)H + (uint32_t)h) * 4u;
            const float3 r3 = load_at<float3>(P.rpos, e * 12u);
            nrx = r3.x; nry = r3.y; nrz = r3.z;
            nz = load_at<float>(C.z, eh); npb = load_at<float>(C.prob, eh);
            nk2 = load_at<float2>(C.k, jh);
            nv2 = load_at<float2>(C.v, jh);
        };
        if (npairs > 0) fetch(0);

        // several chunks: the survivors of all chunks in one list with their index in the whole box (as in the forward)
        const bool one_list = nchunks > 1 && bx.T <= FC_BIGT;
        auto heavy_impl = [&](int nlist, auto big) {
            constexpr bool BIG = decltype(big)::value;      // entries (pair << FC_BIGSHIFT | index in the box), no table
            // (hardware reciprocals, within an ulp: the quotients below stay exact all the same)
            const float inv_s3 = BIG ? hw_rcp((float)bx.s3) : 0.0f, inv_s2 = BIG ? hw_rcp((float)bx.s2) : 0.0f;
            for (int base = 0; base < nlist; base += WAVE) {
                const int idx = base + lane;
                if (idx < nlist) {
                    const uint32_t ent = list[idx];
                    const int pp = BIG ? (int)(ent >> FC_BIGSHIFT) : (int)(ent >> FC_SHIFT);
                    float4 v;
                    if (BIG) {
                        const int tg = (int)(ent & (FC_BIGT - 1));
                        // (exact: the quotients stay below 2^13 and the fractions at least 1 / (2 s) from an integer)
                        const int q = (int)(((float)tg + 0.5f) * inv_s3), i3 = tg - q * bx.s3;
                        const int i1 = (int)(((float)q + 0.5f) * inv_s2), i2 = q - i1 * bx.s2;
                        const float n1 = (float)(i1 - bx.R1), n2 = (float)(i2 - bx.R2), n3 = (float)(i3 - bx.R3);
                        v.x = fmaf(L.t[6], n3, fmaf(L.t[3], n2, L.t[0] * n1));      // as build_shift_table makes them
                        v.y = fmaf(L.t[7], n3, fmaf(L.t[4], n2, L.t[1] * n1));
                        v.z = fmaf(L.t[8], n3, fmaf(L.t[5], n2, L.t[2] * n1));
                        v.w = 0.0f;
                    } else {
                        v = tab[ent & (FC_TCAP - 1)];
                    }
                    const float4 pa = pairA[pp];
                    const float dx = pa.x + v.x, dy = pa.y + v.y, dz = pa.z + v.z;
                    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    const float om = hw_exp2(fmaf(a2, d2, -pa.w)) * pairP[pp];       // P_ij p_n
                    float bg;
                    {
                        const float d = hw_sqrt(d2);
                        const float u = d * bc.inv_interval;
                        int start = (int)(u - bc.start_off);
                        start = max(0, min(start, NBINS - WLr));
                        const float beta_c = ((float)(start + WLr / 2 + 1) - u) * bc.len_step;
                        const WindowSeed s = window_seed(beta_c, bc.len_step, 1.0f);
                        bg = window_gather<WL>(Gs + start, s, bc.len_cc, WLr);
                    }
                    if (HAS_ANG) {
                        if (d2 > 1e-5f) {
                            const float rinv = hw_rsq(d2);
#pragma unroll
                            for (int ax = 0; ax < 3; ax++) {
                                float cs = (dx * f[ax][0] + dy * f[ax][1] + dz * f[ax][2]) * rinv;
                                if (COS_ABS) cs = fabsf(cs);
                                const float uu = (cs - bc.ang_mu0) * bc.ang_inv_interval;
                                if (ANG == SMALL_A) {
                                    const WindowSeed sa = window_seed(((float)(SMALL_A / 2) - uu) * bc.ang_step, bc.ang_step, 1.0f);
                                    bg += window_gather<SMALL_A>(Gs + HW_DIST + ax * SMALL_A, sa, bc.ang_cc);
                                    continue;
                                }
                                const float mf = clampf(__builtin_rintf(uu), 0.0f, (float)(NBINS - 1));
                                const float eps = 2.0f * (uu - mf);
                                const float* gb = Gs + HW_DIST + ax * NORD * NBINS + (int)mf;
                                float pw = eps, part = gb[0];
#pragma unroll
                                for (int o = 1; o < NORD; o++) { part = fmaf(pw, gb[o * NBINS], part); pw *= eps; }
                                bg += part;
                            }
                        }
                    }
                    const float ob = om * bg;
                    cov = fmaf(ob, d2, cov);
                    atomicAdd(pairB + pp, rint_i(ob * bscale));
                }
            }
            n_eval += (unsigned long long)nlist;
        };
        auto heavy = [&](int nlist) { heavy_impl(nlist, std::false_type{}); };

        for (int g0 = 0; g0 < npairs; g0 += FC_GROUP) {
            const float rx = nrx, ry = nry, rz = nrz;
            const float z2 = nz * LOG2E, pij = npb;
            const float2 k2 = nk2, v2 = nv2;
            if (g0 + FC_GROUP < npairs) fetch(g0 + FC_GROUP);
            const bool active = g0 + pr < npairs;
            const float rn = hw_sqrt(fmaf(rx, rx, fmaf(ry, ry, rz * rz)));
            // images with a d^2 log2 e - z2 >= -skip: d^2 <= (z2 - skip) / (a log2 e)
            const float dmax2 = (C.skip_log2 > 0.0f && a2 < 0.0f) ? fmaxf((z2 - C.skip_log2) * inv_a2, 0.0f) : INF;
            const float reach = sorted ? fmaf(1.0001f, rn + hw_sqrt(dmax2), 1e-4f) : FC_REACH_ALL;
            const float lim = active ? fminf(reach, FC_REACH_ALL) : -1.0f;      // (lengths are >= 0; padding: +inf)
            if (lane < FC_GROUP) pairB[lane] = 0;
            if (sub == 0 && active) {
                pairA[pr] = make_float4(rx, ry, rz, z2);
                pairP[pr] = pij;
            }
            float Ap = 0.0f;
            int nlist = 0;
            bool spilled = false;             // (several chunks) more survivors than the list holds: the chunks again, one by one
            if (nchunks == 1) {
                const int cnt = bx.T;
                for (int t0 = 0; t0 < cnt; t0 += FC_GROUP) {
                    const int t = t0 + sub;
                    const float4 v = tab[t];
                    const bool in = v.w <= lim;
                    if (sorted && ballot(in) == 0) break;
                    const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
                    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    const float ex = in ? fmaf(a2, d2, -z2) : -INF;      // (2^-inf = 0, and -inf is below every threshold)
                    Ap = fmaf(hw_exp2(ex), d2, Ap);
                    const bool keep = ex >= prune;
                    const uint64_t m = ballot(keep);
                    if (keep) list[nlist + lane_prefix(m)] = (uint16_t)((pr << FC_SHIFT) | t);
                    nlist += __popcll(m);
                }
            } else {
                for (int ch = 0; ch < nchunks; ch++) {
                    const int t0c = ch * FC_TCAP;
                    const int cnt = min(FC_TCAP, bx.T - t0c);
                    wave_sync();
                    build_shift_table_padded(tab, t0c, cnt, bx, L, lane);
                    wave_sync();
                    for (int t0 = 0; t0 < cnt; t0 += FC_GROUP) {
                        const int t = t0 + sub;
                        const float4 v = tab[t];
                        const bool in = v.w <= lim;
                        const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
                        const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                        const float ex = in ? fmaf(a2, d2, -z2) : -INF;
                        Ap = fmaf(hw_exp2(ex), d2, Ap);
                        if (one_list && !spilled) {
                            const bool keep = ex >= prune;
                            const uint64_t m = ballot(keep);
                            if (nlist + __popcll(m) > FC_LISTCAP) spilled = true;
                            else {
                                if (keep) list[nlist + lane_prefix(m)] = (uint16_t)((pr << FC_BIGSHIFT) | (t0c + t));
                                nlist += __popcll(m);
                            }
                        }
                    }
                }
            }
            const float A0 = half_sum(Ap);
            wave_sync();
            if (nchunks == 1) heavy(nlist);
            else if (one_list && !spilled) heavy_impl(nlist, std::true_type{});
            else {
                for (int ch = 0; ch < nchunks; ch++) {
                    const int t0c = ch * FC_TCAP;
                    const int cnt = min(FC_TCAP, bx.T - t0c);
                    wave_sync();
                    build_shift_table(tab, t0c, cnt, bx, L, lane);
                    wave_sync();
                    int nl = 0;
                    for (int t0 = 0; t0 < cnt; t0 += FC_GROUP) {
                        const int t = t0 + sub;
                        const float4 v = tab[min(t, cnt - 1)];
                        const float dx = rx + v.x, dy = ry + v.y, dz = rz + v.z;
                        const float ex = fmaf(a2, fmaf(dx, dx, fmaf(dy, dy, dz * dz)), -z2);
                        const bool keep = active && t < cnt && ex >= prune;
                        const uint64_t m = ballot(keep);
                        if (keep) list[nl + lane_prefix(m)] = (uint16_t)((pr << FC_SHIFT) | t);
                        nl += __popcll(m);
                    }
                    wave_sync();
                    heavy(nl);
                }
            }
            wave_sync();
            const float gov = half_sum(fmaf(go2.x, v2.x, go2.y * v2.y));          // go . v_j
            const float B1 = (float)pairB[pr] * binv;                             // P_ij (go . psi_ij)
            const float gl = active ? fmaf(pij, gov - c0, B1) : 0.0f;
            gq2.x = fmaf(gl, k2.x, gq2.x);
            gq2.y = fmaf(gl, k2.y, gq2.y);
            if (sub == 0 && active) {
                *reinterpret_cast<float*>(reinterpret_cast<char*>(C.glogit) + ((uint32_t)(e0 + g0 + pr) * (uint32_t)H + (uint32_t)h) * 4u) = gl;
                cov = fmaf(pij * (gov - c0), A0, cov);
            }
            wave_sync();                      // pair data, sums and list may be rewritten
        }
        cov = wave_sum(cov);
        {
            const float gx = rows8_sum(gq2.x), gy = rows8_sum(gq2.y);
            if (lane < FC_GROUP) *reinterpret_cast<float2*>(C.gq + ih * DH + 2 * sub) = make_float2(gx, gy);
        }
        if (lane == 0) P.out_ga[ih] = cov;
        if (P.stats && lane == 0) {
            atomicAdd(P.stats + STAT_BWD_EVAL, n_eval);
            atomicAdd(P.stats + STAT_BWD_RAW, (unsigned long long)bx.T * (unsigned long long)npairs);
            atomicAdd(P.stats + STAT_BWD_PAIRS, (unsigned long long)npairs);
        }
    }
}

}  // namespace cfh
