// What a pass over a batch starts with, in two launches: everything that depends on nothing but the caller's tensors, then
// what is made of it per atom and pair.  The parts are those of geometry.hpp, fused_core.hpp and layer_bridge.hpp; each is
// a few microseconds of work that fills a fraction of the chip.  One by one -- six launches, and a part of every layer's
// launch that makes the item records -- they made up 35 of the 196 us of a call for one crystal; together 15.
#pragma once
#include "fused_core.hpp"
#include "geometry.hpp"
#include "bridge_infer.hpp"

namespace cfh {

constexpr int START_THREADS = GEO_THREADS;
constexpr int START_MAX_WCAT = 24;
struct StartArgs {
    GeometryArgs geo;
    float4* table;                // sorted shifts of every crystal, or null
    int table_R;
    int geo_blocks, table_blocks;      // workgroups of the parts, in this order; behind them the streams
    BridgeStreams streams;
};
// What the second launch makes besides: the cores' concatenated weights, heads x 16 workgroups per layer (the first launch
// has the longer chain without them).
struct StartWcat {
    WcatArgs w[START_MAX_WCAT];
    int n, hc;                    // layers, heads x 16
};
// The prefix sums over the crystals (one workgroup, the longest part) come first.
// (two workgroups per compute unit)
__global__ __launch_bounds__(START_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void model_start_kernel(const StartArgs A) {
    int block = (int)blockIdx.x;
    if (block < A.geo_blocks) { geometry_crystals_block(A.geo, block); return; }
    block -= A.geo_blocks;
    if (block < A.table_blocks) {
        __shared__ float key[START_THREADS];
        constexpr int PER = START_THREADS / FC_TCAP;
        const int sub = (int)threadIdx.x / FC_TCAP;
        const int b = min(block * PER + sub, A.geo.B - 1);      // (past the end: the last crystal again)
        sorted_shifts_block(A.geo.tvecs, A.table_R, A.table, b, (int)threadIdx.x % FC_TCAP, key + sub * FC_TCAP);
        return;
    }
    block -= A.table_blocks;
    const int block256 = block * (START_THREADS / 256) + (int)threadIdx.x / 256, thread = (int)threadIdx.x % 256;
    if (A.streams.split) split_stream_element(A.streams, block256, thread);
    else bridge_stream_element(A.streams, block256, thread);
}
// Workgroups of 256: the concatenated weights, a thread per atom (and one more), eight lanes per pair.
struct PairsArgs {
    GeometryArgs geo;
    float4* table;
    float2* near;
    int table_R, atom_blocks;
};
__global__ __launch_bounds__(256) void model_pairs_kernel(const PairsArgs A, const StartWcat W) {
    int block = (int)blockIdx.x;
    if (block < W.n * W.hc) { core_wcat_block(W.w[block / W.hc], block % W.hc); return; }
    block -= W.n * W.hc;
    const int atom_blocks = A.atom_blocks;
    if (block < atom_blocks) { geometry_atom(A.geo, block * 256 + (int)threadIdx.x); return; }
    const long long e = (long long)(block - atom_blocks) * 32 + (threadIdx.x >> 3);
    const int sub = threadIdx.x & 7;
    PairGeometry g;
    if (!geometry_pair(A.geo, e, g)) return;      // (the same for the eight lanes)
    if (sub == 0) geometry_store_pair(A.geo, e, g);
    if (!A.table) return;
    const int s = 2 * A.table_R + 1;
    const float2 near = pair_nearest(g.x, g.y, g.z, A.table + (size_t)g.crystal * FC_TCAP, s * s * s, sub);
    if (sub == 0) A.near[e] = near;
}

}  // namespace cfh
