// hx_ploc.hip -- PLOC clustering on gfx950 (parallel locally-ordered
// clustering over the Morton-sorted leaves), and the relabelling that turns
// its tree into one whose leaves are numbered in depth-first order, so the
// shared climb and scan-based collapse of hx_build.hip apply unchanged.
//
// Reference (src/hippie/rt/bvh/): PLOCBuilder.cpp:21-208 (clustering loop and
// build), PLOCBuilderKernels.cu:11-113 (generateNeighboursCached), :116-205
// (generateNeighbours), :207-286 (merge), :288-389 (prefix scan + compact).
//
// Per round with m clusters (cluster order = Morton order of the leaves):
//   k_ploc_neighbours  nearest neighbour of every cluster in [i-r, i+r] by the
//                      surface area of the union box; the leftmost minimum
//                      wins (strict '>' over a left-to-right scan);
//   k_ploc_tile_counts merges (mutual pair, lower index) and survivors
//                      (everything but the higher index of a mutual pair) per
//                      512-cluster tile; k_ploc_pairs does both in one
//                      launch for small radii;
//   k_ploc_scan        (rounds of more than kDirectTiles tiles) exclusive scan
//                      of the tile counts, totals for the host;
//   k_ploc_merge       new node = (m-2) - (merge rank in cluster order): the
//                      reference takes this rank from a warp atomicAdd, here it
//                      is a scan so the labels are deterministic; survivors are
//                      written compacted, with their boxes, in cluster order.
// The cluster boxes travel with the clusters (coalesced arrays in cluster
// order), so no round gathers boxes through node indices.
//
// Relabelling (k_tree_down, one launch per round in reverse round order, so
// every parent is placed before its children): offsets of the two children
// from the subtree sizes the merges recorded; a leaf child is renumbered to
// n-1+(its depth-first rank) and its triangle id is written at that rank.
#include <algorithm>
#include <vector>

#include "hx_device.h"
#include "hx_internal.h"

namespace hx {

namespace {

constexpr int kBlock = 256;
// Tile of the flag and merge passes: one cluster per thread.  The passes are
// latency bound (two dependent reads give a flag), so a tile of 16 clusters per
// thread with a block scan each left 244 workgroups of 4 waves for 1,000,003
// clusters; one workgroup of 16 waves per 1024 clusters and ballots instead of
// scans took a round's counts, scan and merge from 43 to 10 us (mean of the 48
// rounds there).  512 for the sake of k_ploc_pairs, whose small rounds then
// spread over more CUs (2310 us with 1024, 2160 with 512, 2175 with 256 for the whole
// build at r = 25; the other radii and 200,003 clusters likewise).
constexpr int kTile = 512;
constexpr int kTileWaves = kTile / kWave;
// Up to this many tiles a merge workgroup adds up the counts before its own
// (at most 64 KB from L2); above it one workgroup scans them first.
constexpr int kDirectTiles = 8192;
constexpr int kPlocBatch = 16;  // rounds launched between host reads
constexpr int kMaxLdsRadius = 1024;   // window of 256 + 2r boxes, 6 floats each, in LDS

inline unsigned grid_for(int64_t n, int block = kBlock) { return (unsigned)((n + block - 1) / block); }

struct Sum2 {
    HX_DEV int2 operator()(int2 a, int2 b) const { return make_int2(a.x + b.x, a.y + b.y); }
};

HX_DEV float3 ld3(const float* p) { return make_float3(p[0], p[1], p[2]); }

// Leaves: box of the sorted triangle p (setupLeaves, LBVHBuilderKernels.cu
// :162-195) as cluster p, node n-1+p.  Also clears what the climb expects
// cleared (counters, cover, frontier count).
__global__ __launch_bounds__(kBlock) void k_ploc_leaves(PlocArgs a) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    const int n = (int)a.n;
    if (p >= n) return;
    Box3 b = box_empty();
    if (a.ref_min) {
        const float4 rmn = a.ref_min[a.sorted_tri[p]], rmx = a.ref_max[a.sorted_tri[p]];
        b.mn = make_float3(rmn.x, rmn.y, rmn.z);
        b.mx = make_float3(rmx.x, rmx.y, rmx.z);
    } else {
        const int32_t* tr = a.tris + 3 * (int64_t)a.sorted_tri[p];
        box_grow(b, ld3(a.verts + 3 * (int64_t)tr[0]));
        box_grow(b, ld3(a.verts + 3 * (int64_t)tr[1]));
        box_grow(b, ld3(a.verts + 3 * (int64_t)tr[2]));
    }
    a.cl[0][p] = n - 1 + p;
    if (a.cm[0]) a.cm[0][p] = a.mesh_of[p];
    a.ca[0][p] = make_float4(b.mn.x, b.mn.y, b.mn.z, b.mx.x);
    a.cb[0][p] = make_float2(b.mx.y, b.mx.z);
    a.end_at[p] = -1;
    if (p < n - 1) a.counters[p] = 0;
    if (p == 0) *a.frontier_count = 0;
}

// area(union) in the reference's order: the neighbour's box grown by the
// cluster's min corner, then by its max corner (AABB::grow, util/AABB.h:26-31).
HX_DEV float union_area(float jx0, float jy0, float jz0, float jx1, float jy1, float jz1, const Box3& own) {
    float mnx = mins(mins(jx0, own.mn.x), own.mx.x), mny = mins(mins(jy0, own.mn.y), own.mx.y);
    float mnz = mins(mins(jz0, own.mn.z), own.mx.z);
    float mxx = maxs(maxs(jx1, own.mn.x), own.mx.x), mxy = maxs(maxs(jy1, own.mn.y), own.mx.y);
    float mxz = maxs(maxs(jz1, own.mn.z), own.mx.z);
    return box_area(make_float3(mnx, mny, mnz), make_float3(mxx, mxy, mxz));
}

// union_area against a cluster known beforehand, halved: lo / hi are the
// component-wise min and max of its two corners.  Cluster boxes hold no NaN
// (they start empty and grow by selects), so min(min(j, mn), mx) =
// min(j, min(mn, mx)), the hardware minimum differs from the select only in
// the sign of a zero, which no comparison of areas sees, and the union is
// always valid; without the factor 2 (exact, and the start value is halved
// too) the order of areas is the same.  Six min/max instead of twelve selects
// (24 instructions) a pair.
HX_DEV float vmin(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
HX_DEV float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
constexpr float kHalfMax = 0.5f * kMaxFloat;
HX_DEV float half_union_area(float4 x, float2 y, float3 lo, float3 hi) {
    const float dx = vmax(x.w, hi.x) - vmin(x.x, lo.x);
    const float dy = vmax(y.x, hi.y) - vmin(x.y, lo.y);
    const float dz = vmax(y.y, hi.z) - vmin(x.z, lo.z);
    return dx * dy + dy * dz + dz * dx;
}
// A box no cluster can be nearest to: every union with it has an infinite
// area (MAX - -MAX overflows).
HX_DEV float4 far_box_a() { return make_float4(-kMaxFloat, -kMaxFloat, -kMaxFloat, kMaxFloat); }
HX_DEV float2 far_box_b() { return make_float2(kMaxFloat, kMaxFloat); }

HX_DEV Box3 cluster_box(float4 a, float2 b) {
    Box3 r;
    r.mn = make_float3(a.x, a.y, a.z);
    r.mx = make_float3(a.w, b.x, b.y);
    return r;
}

// Nearest cluster of i within [i - r, i + r] (same mesh if cmesh), the
// lowest index on ties, from global memory.
HX_DEV int nearest_cluster(const float4* __restrict__ ca, const float2* __restrict__ cb, int m, int r, int i,
                           const int32_t* __restrict__ cmesh) {
    const Box3 own = cluster_box(ca[i], cb[i]);
    int best = -1;
    float bestD = kMaxFloat;
    const int jlo = max(0, i - r), jhi = min(m - 1, i + r);
    const int mine = cmesh ? cmesh[i] : 0;
    for (int j = jlo; j <= jhi; ++j) {
        if (j == i) continue;
        if (cmesh && cmesh[j] != mine) continue;
        const float4 x = ca[j];
        const float2 y = cb[j];
        const float d = union_area(x.x, x.y, x.z, x.w, y.x, y.y, own);
        if (bestD > d) {
            bestD = d;
            best = j;
        }
    }
    return best;
}

// The round's cluster count m is read from its record (rounds run ahead of the
// host); a finished build (m <= 1) makes the round a no-op.  Batched builds
// pass the cluster mesh ids: a cluster only looks at clusters of its own mesh
// (the meshes' cluster runs are contiguous, so this is the single-mesh window
// clipped to the mesh), and once every mesh is one cluster (m <= n_meshes) the
// round pairs clusters (2k, 2k+1) instead (see launch_ploc).
HX_DEV bool ploc_pair_round(int m, const int32_t* cmesh, int n_meshes, int i, int32_t* nb) {
    if (!cmesh || m > n_meshes) return false;
    if (i < m) nb[i] = (i ^ 1) < m ? (i ^ 1) : -1;
    return true;
}

// Place of the cluster nearest to the one at place `me` among the places [q0, q1)
// (the lowest on ties), -1 without one; sa, sb: boxes, sm: meshes.
template <bool MESH>
HX_DEV int scan_window(const float4* sa, const float2* sb, const int32_t* sm, int me, int q0, int q1) {
    const Box3 own = cluster_box(sa[me], sb[me]);
    const float3 lo = make_float3(vmin(own.mn.x, own.mx.x), vmin(own.mn.y, own.mx.y), vmin(own.mn.z, own.mx.z));
    const float3 hi = make_float3(vmax(own.mn.x, own.mx.x), vmax(own.mn.y, own.mx.y), vmax(own.mn.z, own.mx.z));
    const int mine = MESH ? sm[me] : 0;
    int best = -1;
    float bestD = kHalfMax;
    auto step = [&](int q) {
        const float d = half_union_area(sa[q], sb[q], lo, hi);
        const bool better = bestD > d && (!MESH || sm[q] == mine);
        bestD = better ? d : bestD;
        best = better ? q : best;
    };
    auto scan = [&](int q, int end) {
        for (; q + 4 <= end; q += 4) {
            step(q);
            step(q + 1);
            step(q + 2);
            step(q + 3);
        }
        for (; q < end; ++q) step(q);
    };
    scan(q0, me);
    scan(me + 1, q1);
    return best;
}

// The window [b0 - r, b0 + kBlock + r) of a workgroup's clusters in LDS, places
// outside [0, m) filled with far boxes, so that every lane scans the same 2r
// places with no bounds tests.  VALU bound: 17 instructions and two LDS reads
// (16 + 8 bytes) a pair instead of 35 and six; the 48 rounds of a 1,000,003-triangle
// build at r = 25 went from 937 to 375 us.
template <bool MESH>
__global__ __launch_bounds__(kBlock) void k_ploc_neighbours(const float4* __restrict__ ca,
                                                            const float2* __restrict__ cb,
                                                            const int4* __restrict__ round, int r,
                                                            int32_t* __restrict__ nb,
                                                            const int32_t* __restrict__ cmesh, int n_meshes) {
    extern __shared__ float4 s_win[];
    const int W = kBlock + 2 * r;
    float4* sa = s_win;
    float2* sb = reinterpret_cast<float2*>(sa + W);
    int32_t* sm = reinterpret_cast<int32_t*>(sb + W);
    const int m = round->x;
    const int b0 = blockIdx.x * kBlock;
    const int i = b0 + threadIdx.x;
    if (m <= 1 || b0 >= m) return;
    if (MESH && ploc_pair_round(m, cmesh, n_meshes, i, nb)) return;
    for (int k = threadIdx.x; k < W; k += kBlock) {
        const int j = b0 - r + k;
        const bool in = j >= 0 && j < m;
        sa[k] = in ? ca[j] : far_box_a();
        sb[k] = in ? cb[j] : far_box_b();
        if (MESH) sm[k] = in ? cmesh[j] : -1;
    }
    __syncthreads();
    if (i >= m) return;
    const int best = scan_window<MESH>(sa, sb, sm, threadIdx.x + r, threadIdx.x, threadIdx.x + 2 * r + 1);
    nb[i] = best < 0 ? -1 : best + b0 - r;
}

// Windows that do not fit in LDS (r > kMaxLdsRadius).
__global__ __launch_bounds__(kBlock) void k_ploc_neighbours_far(const float4* __restrict__ ca,
                                                                const float2* __restrict__ cb,
                                                                const int4* __restrict__ round, int r,
                                                                int32_t* __restrict__ nb,
                                                                const int32_t* __restrict__ cmesh, int n_meshes) {
    const int m = round->x;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (m <= 1 || i >= m || ploc_pair_round(m, cmesh, n_meshes, i, nb)) return;
    nb[i] = nearest_cluster(ca, cb, m, r, i, cmesh);
}

// (merging, surviving) of cluster i (PLOCBuilderKernels.cu:232-240): -- a mutual pair merges
// into the lower index; the higher index drops out of the compacted list.
HX_DEV int2 ploc_flags(const int32_t* __restrict__ nb, int m, int64_t i) {
    if (i >= m) return make_int2(0, 0);
    const int j = nb[i];
    const bool mutual = j >= 0 && nb[j] == (int)i;
    return make_int2(mutual && i < j ? 1 : 0, (mutual && i > j) ? 0 : 1);
}

// Merging and surviving clusters of a workgroup's tile per wave (ws), from
// ballots; every thread of the workgroup calls it.
HX_DEV void tile_ballots(int2 f, uint64_t& bm, uint64_t& bs, int2* ws) {
    bm = ballot64(f.x != 0);
    bs = ballot64(f.y != 0);
    if (lane_id() == 0) ws[threadIdx.x / kWave] = make_int2(__popcll(bm), __popcll(bs));
    __syncthreads();
}

// The sum of the waves' counts of tile_ballots, by one thread.
HX_DEV int2 tile_sum(const int2* ws) {
    int2 s = ws[0];
    for (int w = 1; w < kTileWaves; ++w) s = make_int2(s.x + ws[w].x, s.y + ws[w].y);
    return s;
}

// Neighbours and tile counts in one launch.  The kTile threads find the
// neighbours of the tile's kTile - 2r clusters and of the r clusters on either
// side, so that the tile's mutual pairs are known from LDS alone.  Most rounds
// are too small to take longer than a launch, and this saves one of three;
// the work grows by kTile / (kTile - 2r), so larger radii and rounds keep two
// kernels.  Builds of 1,000,003 triangles, two kernels and one: r = 8 1725 and
// 1624 us, r = 25 2290 and 2165, r = 48 2745 and 2675, r = 64 3033 and 3021;
// 16.7M triangles at r = 25 18.50 and 18.64 ms.
constexpr int kFusedRadius = 48;
constexpr int kFusedClusters = 1 << 22;
template <bool MESH>
__global__ __launch_bounds__(kTile) void k_ploc_pairs(const float4* __restrict__ ca, const float2* __restrict__ cb,
                                                      const int4* __restrict__ round, int r,
                                                      int32_t* __restrict__ nb, const int32_t* __restrict__ cmesh,
                                                      int n_meshes, int2* __restrict__ partial) {
    extern __shared__ float4 s_win[];
    __shared__ int s_nb[kTile];
    __shared__ int2 ws[kTileWaves];
    const int W = kTile + 2 * r;
    float4* sa = s_win;
    float2* sb = reinterpret_cast<float2*>(sa + W);
    int32_t* sm = reinterpret_cast<int32_t*>(sb + W);
    const int m = round->x;
    const int b0 = blockIdx.x * (kTile - 2 * r);
    if (m <= 1 || b0 >= m) return;
    const int t = threadIdx.x;
    const int i = b0 - r + t;  // this thread's cluster, if 0 <= i < m
    int j = -1;
    if (MESH && m <= n_meshes) {
        if (i >= 0 && i < m && (i ^ 1) < m) j = i ^ 1;  // ploc_pair_round
    } else {
        for (int k = t; k < W; k += kTile) {
            const int q = b0 - 2 * r + k;
            const bool in = q >= 0 && q < m;
            sa[k] = in ? ca[q] : far_box_a();
            sb[k] = in ? cb[q] : far_box_b();
            if (MESH) sm[k] = in ? cmesh[q] : -1;
        }
        __syncthreads();
        if (i >= 0 && i < m) {
            const int best = scan_window<MESH>(sa, sb, sm, t + r, t, t + 2 * r + 1);
            j = best < 0 ? -1 : best + b0 - 2 * r;
        }
    }
    s_nb[t] = j;
    __syncthreads();
    const bool own = t >= r && t < kTile - r && i < m;
    const bool mutual = own && j >= 0 && s_nb[j - (b0 - r)] == i;
    if (own) nb[i] = j;
    uint64_t bm, bs;
    tile_ballots(make_int2(mutual && i < j ? 1 : 0, own && !(mutual && i > j) ? 1 : 0), bm, bs, ws);
    if (t == 0) partial[blockIdx.x] = tile_sum(ws);
}

__global__ __launch_bounds__(kTile) void k_ploc_tile_counts(const int32_t* __restrict__ nb,
                                                            const int4* __restrict__ round,
                                                            int2* __restrict__ partial) {
    __shared__ int2 ws[kTileWaves];
    const int m = round->x;
    const int64_t base = blockIdx.x * (int64_t)kTile;
    if (m <= 1 || base >= m) return;
    uint64_t bm, bs;
    tile_ballots(ploc_flags(nb, m, base + threadIdx.x), bm, bs, ws);
    if (threadIdx.x == 0) partial[blockIdx.x] = tile_sum(ws);
}

// The round's totals (merged, surviving) to its record, whose cluster count
// other workgroups may still be reading; the survivors are the next round's
// clusters.
HX_DEV void close_round(int4* round, int2 tot) {
    round->y = tot.x;
    round->z = tot.y;
    round[1] = make_int4(tot.y, 0, 0, 0);
}

// Single block: exclusive scan of the tile counts in place; the round's
// (merged, surviving) totals go to its record and the survivors become the
// next round's cluster count.
__global__ __launch_bounds__(kTile) void k_ploc_scan(int2* __restrict__ partial, int4* __restrict__ round,
                                                     int tile_size) {
    __shared__ int2 wt[kTileWaves];
    const int m = round->x;
    if (m <= 1) {
        if (threadIdx.x == 0) close_round(round, make_int2(0, m));
        return;
    }
    const int ntiles = (m + tile_size - 1) / tile_size;
    int2 carry = make_int2(0, 0);
    for (int base = 0; base < ntiles; base += kTile) {
        const int t = base + threadIdx.x;
        const int2 v = t < ntiles ? partial[t] : make_int2(0, 0);
        int2 tot;
        const int2 inc = block_inclusive_scan<kTileWaves>(v, Sum2(), wt, tot);
        if (t < ntiles) partial[t] = make_int2(carry.x + inc.x - v.x, carry.y + inc.y - v.y);
        carry = make_int2(carry.x + tot.x, carry.y + tot.y);
    }
    if (threadIdx.x == 0) close_round(round, carry);
}

// Cluster i of a round with flags f (merging, surviving) and ranks among the
// merging and surviving clusters: a merging cluster creates node
// node_offset - mrank from itself and its neighbour; survivors move to slot
// srank of the other cluster buffer.
HX_DEV void merge_cluster(const PlocArgs& a, int src, int i, int2 f, int mrank, int srank, int node_offset) {
    const int n = (int)a.n;
    const int32_t* __restrict__ cl = a.cl[src];
    const float4* __restrict__ ca = a.ca[src];
    const float2* __restrict__ cb = a.cb[src];
    int32_t* __restrict__ cl_out = a.cl[src ^ 1];
    float4* __restrict__ ca_out = a.ca[src ^ 1];
    float2* __restrict__ cb_out = a.cb[src ^ 1];
    if (f.x) {
        const int j = a.nb[i];
        const int ln = cl[i], rn = cl[j];
        const int node = node_offset - mrank;
        const Box3 lb = cluster_box(ca[i], cb[i]);
        const Box3 rb = cluster_box(ca[j], cb[j]);
        a.parent[ln] = node;
        a.parent[rn] = node;
        a.left[node] = ln;
        a.right[node] = rn;
        const int sl = ln >= n - 1 ? 1 : a.last[ln];
        const int sr = rn >= n - 1 ? 1 : a.last[rn];
        a.last[node] = sl + sr;
        cl_out[srank] = node;
        if (a.cm[0]) a.cm[src ^ 1][srank] = a.cm[src][i];
        ca_out[srank] = make_float4(mins(lb.mn.x, rb.mn.x), mins(lb.mn.y, rb.mn.y), mins(lb.mn.z, rb.mn.z),
                                    maxs(lb.mx.x, rb.mx.x));
        cb_out[srank] = make_float2(maxs(lb.mx.y, rb.mx.y), maxs(lb.mx.z, rb.mx.z));
    } else if (f.y) {
        cl_out[srank] = cl[i];
        if (a.cm[0]) a.cm[src ^ 1][srank] = a.cm[src][i];
        ca_out[srank] = ca[i];
        cb_out[srank] = cb[i];
    }
}

// merge (PLOCBuilderKernels.cu:207-286) + compact (:288-389) in one pass.
// The new node's box is the select-based union of the two cluster boxes
// (the reference uses fminf/fmaxf, which differ from selects only in the sign
// of a zero); its subtree size goes to last[node] for the relabelling.
// SCANNED: partial holds exclusive prefixes (k_ploc_scan); else the counts, which
// the workgroup adds up itself, and the workgroup of the last tile closes the
// round.  tile_size: clusters of a tile, as the counts were taken.
template <bool SCANNED>
__global__ __launch_bounds__(kTile) void k_ploc_merge(PlocArgs a, int src, int4* __restrict__ round,
                                                      const int2* __restrict__ partial, int tile_size) {
    __shared__ int2 ws[kTileWaves], pre[kTileWaves];
    const int m = round->x;
    const int tile = blockIdx.x;
    const int64_t base = tile * (int64_t)tile_size;
    if (m <= 1) {
        if (!SCANNED && tile == 0 && threadIdx.x == 0) close_round(round, make_int2(0, m));
        return;
    }
    if (base >= m) return;
    const int64_t i = (int)threadIdx.x < tile_size ? base + threadIdx.x : m;
    const int2 f = ploc_flags(a.nb, m, i);
    const int w = threadIdx.x / kWave;
    int2 carry = make_int2(0, 0);
    if (SCANNED) {
        carry = partial[tile];
    } else {
        int2 s = make_int2(0, 0);
        for (int t = threadIdx.x; t < tile; t += kTile) s = make_int2(s.x + partial[t].x, s.y + partial[t].y);
        s = make_int2(wave_sum_i32(s.x), wave_sum_i32(s.y));
        if (lane_id() == 0) pre[w] = s;
    }
    uint64_t bm, bs;
    tile_ballots(f, bm, bs, ws);
    int2 tot = make_int2(0, 0), below = make_int2(0, 0);
#pragma unroll
    for (int k = 0; k < kTileWaves; ++k) {
        if (!SCANNED) carry = make_int2(carry.x + pre[k].x, carry.y + pre[k].y);
        if (k == w) below = tot;
        tot = make_int2(tot.x + ws[k].x, tot.y + ws[k].y);
    }
    if (i < m)
        merge_cluster(a, src, (int)i, f, carry.x + below.x + count_below(bm), carry.y + below.y + count_below(bs), m - 2);
    if (!SCANNED && base + tile_size >= m && threadIdx.x == 0)
        close_round(round, make_int2(carry.x + tot.x, carry.y + tot.y));
}

__global__ void k_ploc_round_start(int4* round, int m) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *round = make_int4(m, 0, 0, 0);
}

// The last rounds (at most kTailClusters clusters) in one workgroup, with three
// barriers a round instead of three launches.  The clusters (boxes, ids,
// subtree sizes, mesh ids) and their neighbours stay in LDS from the first
// round to the last; each thread holds at most two of them, ranks them from
// ballots and writes the survivors back in place once every thread has read
// its pair.  rec[k] = (clusters, merged, surviving) of tail round k; *nrec =
// rounds run (a round that merges nothing ends it).  Staging each round from
// global memory, with flags read back from there, took 571 us for the last
// 2048 clusters of a 1,000,003-triangle build; this form takes 181 us.
constexpr int kTailBlock = 1024;
constexpr int kTailClusters = 2048;
constexpr int kTailWaves = kTailBlock / kWave;

template <bool BATCHED>
__global__ __launch_bounds__(kTailBlock) void k_ploc_tail(PlocArgs a, int src, int m, int r, int4* __restrict__ rec,
                                                          int* __restrict__ nrec) {
    constexpr int kPer = kTailClusters / kTailBlock;
    __shared__ float4 s_a[kTailClusters];
    __shared__ float2 s_b[kTailClusters];
    __shared__ int s_id[kTailClusters], s_size[kTailClusters], s_nb[kTailClusters];
    __shared__ int s_mesh[BATCHED ? kTailClusters : 1];
    __shared__ int2 s_cnt[kPer][kTailWaves];
    const int n = (int)a.n;
    const int t = threadIdx.x, w = t / kWave;
    for (int i = t; i < m; i += kTailBlock) {
        s_a[i] = a.ca[src][i];
        s_b[i] = a.cb[src][i];
        const int id = a.cl[src][i];
        s_id[i] = id;
        s_size[i] = id >= n - 1 ? 1 : a.last[id];
        if (BATCHED) s_mesh[i] = a.cm[src][i];
    }
    int k = 0;
    while (m > 1) {
        if (a.adaptive) r = min(r + 1, a.max_radius);
        const bool pairs = BATCHED && m <= a.n_meshes;
        __syncthreads();
        for (int i = t; i < m; i += kTailBlock) {
            if (pairs) {
                s_nb[i] = (i ^ 1) < m ? (i ^ 1) : -1;
                continue;
            }
            s_nb[i] = scan_window<BATCHED>(s_a, s_b, s_mesh, i, max(0, i - r), min(m, i + r + 1));
        }
        __syncthreads();
        int2 f[kPer];
        uint64_t bm[kPer], bs[kPer];
        float4 oa[kPer];
        float2 ob[kPer];
        int ol[kPer], orr[kPer], osz[kPer], om[kPer];
#pragma unroll
        for (int p = 0; p < kPer; ++p) {
            const int i = t + p * kTailBlock;
            f[p] = make_int2(0, 0);
            oa[p] = make_float4(0.f, 0.f, 0.f, 0.f);
            ob[p] = make_float2(0.f, 0.f);
            ol[p] = orr[p] = -1;
            osz[p] = om[p] = 0;
            if (i < m) {
                const int j = s_nb[i];
                const bool mutual = j >= 0 && s_nb[j] == i;
                f[p] = make_int2(mutual && i < j ? 1 : 0, mutual && i > j ? 0 : 1);
                oa[p] = s_a[i];
                ob[p] = s_b[i];
                ol[p] = s_id[i];
                osz[p] = s_size[i];
                if (BATCHED) om[p] = s_mesh[i];
                if (f[p].x) {
                    const float4 x = s_a[j];
                    const float2 y = s_b[j];
                    oa[p] = make_float4(mins(oa[p].x, x.x), mins(oa[p].y, x.y), mins(oa[p].z, x.z), maxs(oa[p].w, x.w));
                    ob[p] = make_float2(maxs(ob[p].x, y.x), maxs(ob[p].y, y.y));
                    orr[p] = s_id[j];
                    osz[p] += s_size[j];
                }
            }
            bm[p] = ballot64(f[p].x != 0);
            bs[p] = ballot64(f[p].y != 0);
            if (lane_id() == 0) s_cnt[p][w] = make_int2(__popcll(bm[p]), __popcll(bs[p]));
        }
        __syncthreads();
        int2 tot = make_int2(0, 0), below[kPer];
#pragma unroll
        for (int p = 0; p < kPer; ++p) {
            below[p] = make_int2(0, 0);
            for (int q = 0; q < kTailWaves; ++q) {
                if (q == w) below[p] = tot;
                tot = make_int2(tot.x + s_cnt[p][q].x, tot.y + s_cnt[p][q].y);
            }
        }
        if (t == 0) rec[k] = make_int4(m, tot.x, tot.y, 0);
        ++k;
        if (tot.x == 0) break;
#pragma unroll
        for (int p = 0; p < kPer; ++p) {
            if (!f[p].y) continue;  // dropped, or past the end
            const int slot = below[p].y + count_below(bs[p]);
            int id = ol[p];
            if (f[p].x) {
                id = m - 2 - (below[p].x + count_below(bm[p]));
                a.parent[ol[p]] = id;
                a.parent[orr[p]] = id;
                a.left[id] = ol[p];
                a.right[id] = orr[p];
                a.last[id] = osz[p];
            }
            s_a[slot] = oa[p];
            s_b[slot] = ob[p];
            s_id[slot] = id;
            s_size[slot] = osz[p];
            if (BATCHED) s_mesh[slot] = om[p];
        }
        m = tot.y;
    }
    if (t == 0) *nrec = k;
}

// Depth-first placement of the children of the nodes list[0, count) (or, if
// list is NULL, of lo + [0, count)), all independent: every parent was placed
// by an earlier launch.  last[v] holds v's subtree size on entry and its last
// leaf rank on exit; first[v] was written by v's parent (the root starts at 0).
HX_DEV void tree_down_node(const PlocArgs& a, int v) {
    const int n = (int)a.n;
    const int off = v == 0 ? 0 : a.first[v];
    const int size = a.last[v];
    const int l = a.left[v], r = a.right[v];
    const int sl = l >= n - 1 ? 1 : a.last[l];
    if (v == 0) {
        a.first[0] = 0;
        a.parent[0] = -1;
    }
    a.last[v] = off + size - 1;
    a.split[v] = off + sl - 1;
    const int ch[2] = {l, r};
    const int co[2] = {off, off + sl};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int c = ch[k], o = co[k];
        // A consistent tree keeps every index in range; a broken one must not
        // write outside the arrays.
        if ((unsigned)c >= (unsigned)(2 * n - 1) || (unsigned)o >= (unsigned)n) continue;
        if (c >= n - 1) {
            const int leaf = n - 1 + o;
            a.tri_out[o] = a.sorted_tri[c - (n - 1)];
            a.parent[leaf] = v;
            a.first[leaf] = o;
            a.last[leaf] = o;
            a.left[leaf] = o;
            a.right[leaf] = o + 1;
            if (k == 0)
                a.left[v] = leaf;
            else
                a.right[v] = leaf;
        } else {
            a.first[c] = o;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_tree_down(PlocArgs a, const int32_t* __restrict__ list, int lo,
                                                      int count) {
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    tree_down_node(a, list ? list[k] : lo + k);
}

// Several placement steps in one workgroup, a barrier between steps (the
// barrier orders the global writes of a step before the next step's reads
// within the workgroup).
constexpr int kStepBlock = 1024;
constexpr int kSmallStep = 4 * kStepBlock;  // steps up to this many nodes share the workgroup

__global__ __launch_bounds__(kStepBlock) void k_tree_down_steps(PlocArgs a, const int32_t* __restrict__ list,
                                                                const int2* __restrict__ segs, int nsegs) {
    for (int k = 0; k < nsegs; ++k) {
        const int2 sg = segs[k];
        for (int j = threadIdx.x; j < sg.y; j += kStepBlock) tree_down_node(a, list ? list[sg.x + j] : sg.x + j);
        __syncthreads();
    }
}

}  // namespace

int launch_tree_down_steps(Context* c, const PlocArgs& a, const int32_t* list, const std::vector<int2>& segs) {
    size_t small = 0;
    while (small < segs.size() && segs[small].y <= kSmallStep) ++small;
    if (small > 1) {
        HX_TRY(c->segments.reserve(sizeof(int2) * small));
        c->segments_host.assign(segs.begin(), segs.begin() + small);
        HX_HIP(hipMemcpyAsync(c->segments.ptr, c->segments_host.data(), sizeof(int2) * small, hipMemcpyHostToDevice,
                              c->stream));
        hipLaunchKernelGGL(k_tree_down_steps, dim3(1), dim3(kStepBlock), 0, c->stream, a, list,
                           c->segments.as<int2>(), (int)small);
        HX_TRY(check_launch("tree_down_steps"));
    } else {
        small = 0;
    }
    for (size_t k = small; k < segs.size(); ++k) {
        if (segs[k].y <= 0) continue;
        hipLaunchKernelGGL(k_tree_down, dim3(grid_for(segs[k].y)), dim3(kBlock), 0, c->stream, a,
                           list ? list + segs[k].x : nullptr, list ? 0 : segs[k].x, segs[k].y);
        HX_TRY(check_launch("tree_down"));
    }
    return HX_OK;
}

int launch_ploc(Context* c, const PlocArgs& a, int* rounds_out) {
    const int n = (int)a.n;
    {
        LaunchScope ls(c, "ploc_leaves");
        hipLaunchKernelGGL(k_ploc_leaves, dim3(grid_for(n)), dim3(kBlock), 0, c->stream, a);
        HX_TRY(check_launch("ploc_leaves"));
    }
    constexpr int kMinTile = kTile - 2 * kFusedRadius;
    const int64_t max_tiles = (n + kMinTile - 1) / kMinTile;
    HX_TRY(c->scan_partials.reserve(sizeof(int2) * (size_t)max_tiles + sizeof(int4) * (kPlocBatch + kTailClusters + 2) +
                                    64));
    int2* partial = c->scan_partials.as<int2>();
    int4* rounds = reinterpret_cast<int4*>(partial + ((max_tiles + 1) & ~(int64_t)1));
    int4* tail_rec = rounds + kPlocBatch + 1;
    int* tail_count = reinterpret_cast<int*>(tail_rec + kTailClusters);
    std::vector<int2> ranges;   // [lo, hi] of the nodes each round created
    // Batched builds merge inside each mesh until every mesh is one cluster
    // (m == n_meshes), then join the mesh roots pairwise in mesh order
    // (separators, never emitted), so mesh m's leaves keep positions
    // [off[m], off[m+1]) after the depth-first relabelling.
    const bool batched = a.cm[0] != nullptr && a.n_meshes > 1;
    // Rounds run on the device in batches of kPlocBatch: each reads its cluster
    // count from the previous round's record, and the host reads the records
    // once per batch (grids are sized by the count known at the batch start).
    int m = n, src = 0, r = a.radius;
    std::vector<int4> h_rounds(kPlocBatch + 1);
    hipLaunchKernelGGL(k_ploc_round_start, dim3(1), dim3(64), 0, c->stream, rounds, m);
    HX_TRY(check_launch("ploc_round_start"));
    while (m > 1) {
        if (m <= kTailClusters) {
            LaunchScope ls(c, "ploc_tail");
            hipLaunchKernelGGL((batched ? k_ploc_tail<true> : k_ploc_tail<false>), dim3(1), dim3(kTailBlock), 0,
                               c->stream, a, src, m, r, tail_rec, tail_count);
            HX_TRY(check_launch("ploc_tail"));
            int cnt = 0;
            HX_HIP(hipMemcpyAsync(&cnt, tail_count, sizeof(int), hipMemcpyDeviceToHost, c->stream));
            HX_HIP(hipStreamSynchronize(c->stream));
            std::vector<int4> rec((size_t)std::max(cnt, 0));
            if (cnt > 0) {
                HX_HIP(hipMemcpyAsync(rec.data(), tail_rec, sizeof(int4) * rec.size(), hipMemcpyDeviceToHost,
                                      c->stream));
                HX_HIP(hipStreamSynchronize(c->stream));
            }
            for (const int4& t : rec) {
                if (t.y <= 0 || t.y + t.z != t.x) {
                    set_error("PLOC round with %d clusters merged %d pairs (non-finite boxes?)", t.x, t.y);
                    return HX_ERR_INVALID_ARG;
                }
                ranges.push_back(make_int2(t.x - 2 - t.y + 1, t.x - 2));
            }
            break;
        }
        for (int b = 0; b < kPlocBatch; ++b) {
            if (a.adaptive) r = std::min(r + 1, a.max_radius);
            const int32_t* cmesh = batched ? a.cm[src] : nullptr;
            const bool fused = r <= kFusedRadius && m <= kFusedClusters;
            const int tile_size = fused ? kTile - 2 * r : kTile;
            const int ntiles = (m + tile_size - 1) / tile_size;
            {
                LaunchScope ls(c, "ploc_neighbours");
                const size_t lds = sizeof(float) * (batched ? 7 : 6) * (size_t)((fused ? kTile : kBlock) + 2 * r);
                if (fused) {
                    hipLaunchKernelGGL((batched ? k_ploc_pairs<true> : k_ploc_pairs<false>), dim3(ntiles), dim3(kTile),
                                       lds, c->stream, a.ca[src], a.cb[src], rounds + b, r, a.nb, cmesh, a.n_meshes,
                                       partial);
                    HX_TRY(check_launch("ploc_pairs"));
                } else {
                    auto kernel = r > kMaxLdsRadius ? k_ploc_neighbours_far
                                                    : batched ? k_ploc_neighbours<true> : k_ploc_neighbours<false>;
                    hipLaunchKernelGGL(kernel, dim3(grid_for(m)), dim3(kBlock), r > kMaxLdsRadius ? 0 : lds, c->stream,
                                       a.ca[src], a.cb[src], rounds + b, r, a.nb, cmesh, a.n_meshes);
                    HX_TRY(check_launch("ploc_neighbours"));
                }
            }
            {
                LaunchScope ls(c, "ploc_merge");
                if (!fused) {
                    hipLaunchKernelGGL(k_ploc_tile_counts, dim3(ntiles), dim3(kTile), 0, c->stream, a.nb, rounds + b,
                                       partial);
                    HX_TRY(check_launch("ploc_tile_counts"));
                }
                const bool direct = ntiles <= kDirectTiles;
                if (!direct) {
                    hipLaunchKernelGGL(k_ploc_scan, dim3(1), dim3(kTile), 0, c->stream, partial, rounds + b,
                                       tile_size);
                    HX_TRY(check_launch("ploc_scan"));
                }
                hipLaunchKernelGGL((direct ? k_ploc_merge<false> : k_ploc_merge<true>), dim3(ntiles), dim3(kTile), 0,
                                   c->stream, a, src, rounds + b, partial, tile_size);
                HX_TRY(check_launch("ploc_merge"));
            }
            src ^= 1;
        }
        HX_HIP(hipMemcpyAsync(h_rounds.data(), rounds, sizeof(int4) * h_rounds.size(), hipMemcpyDeviceToHost,
                              c->stream));
        HX_HIP(hipStreamSynchronize(c->stream));
        for (int b = 0; b < kPlocBatch; ++b) {
            const int4 t = h_rounds[b];
            if (t.x <= 1) break;
            if (t.y <= 0 || t.y + t.z != t.x) {
                set_error("PLOC round with %d clusters merged %d pairs (non-finite boxes?)", t.x, t.y);
                return HX_ERR_INVALID_ARG;
            }
            ranges.push_back(make_int2(t.x - 2 - t.y + 1, t.x - 2));
        }
        m = h_rounds[kPlocBatch].x;
        if (m > 1) {
            hipLaunchKernelGGL(k_ploc_round_start, dim3(1), dim3(64), 0, c->stream, rounds, m);
            HX_TRY(check_launch("ploc_round_start"));
        }
    }
    {
        LaunchScope ls(c, "ploc_relabel");
        std::vector<int2> segs;  // rounds in reverse order: parents first
        for (size_t k = ranges.size(); k-- > 0;) segs.push_back(make_int2(ranges[k].x, ranges[k].y - ranges[k].x + 1));
        HX_TRY(launch_tree_down_steps(c, a, nullptr, segs));
    }
    if (rounds_out) *rounds_out = (int)ranges.size();
    return HX_OK;
}

}  // namespace hx
