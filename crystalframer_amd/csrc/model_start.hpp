// What a pass over a batch starts with, in two launches: everything that depends on nothing but the caller's tensors, then
// what is made of it per atom and pair.  The parts are those of geometry.hpp, fused_core.hpp and layer_bridge.hpp; each is
// a few microseconds of work that fills a fraction of the chip, and one by one -- five launches, and a part of every layer's
// launch that makes the item records -- they took @@.
#pragma once
#include "fused_core.hpp"
#include "geometry.hpp"
#include "layer_bridge.hpp"

namespace cfh {

constexpr int START_THREADS = GEO_THREADS;
constexpr int START_MAX_WCAT = 8;
struct StartArgs {
    GeometryArgs geo;
    float4* table;                // sorted shifts of every crystal, or null
    float2* near;                 // nearest images of every pair over that table
    int table_R;
    int geo_blocks, table_blocks, stream_blocks;      // workgroups of the parts, in this order; then heads x 16 per layer
    int hc;                       // heads x 16
    BridgeStreams streams;
    WcatArgs wcat[START_MAX_WCAT];
};
// The prefix sums over the crystals (one workgroup, the longest part) come first.
__global__ __launch_bounds__(START_THREADS) void model_start_kernel(const StartArgs A) {
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
    if (block < A.stream_blocks) {
        bridge_stream_element(A.streams, block * (START_THREADS / 256) + (int)threadIdx.x / 256, (int)threadIdx.x % 256);
        return;
    }
    block -= A.stream_blocks;
    core_wcat_block(A.wcat[block / A.hc], block % A.hc);
}
// Workgroups of 256: a thread per atom (and one more), then eight lanes per pair.
__global__ __launch_bounds__(256) void model_pairs_kernel(const StartArgs A, int atom_blocks) {
    const int block = (int)blockIdx.x;
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
