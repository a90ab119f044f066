// hx_atr.hip -- ATRBVH (agglomerative treelet restructuring) on gfx950.
//
// Reference (src/hippie/rt/bvh/): ATRBuilder.cpp:23-236 (schedule, optimise
// loop, build), ATRBuilderKernels.cu:11-577 (optimize / optimizeSmall and
// their helpers), TRBuilderUtil.h:11-289 (formTreelet and the area helpers).
//
// The reference climbs from every leaf with atomic counters, recomputes every
// node's cost on the way, and lets a 32-lane warp restructure each node whose
// subtree holds at least gamma references.  Here the climb order is replaced by
// a level order: before each iteration the internal nodes are bucketed by
// (subtree height, >= gamma references), and per height one launch recomputes
// the costs of the small nodes (a thread each) and one restructures the large
// ones (32 lanes each).  Nodes of one height are never ancestors of each other
// and each treelet lies inside its root's subtree, so a height's nodes are
// independent, and every parent is processed after its children as in the
// reference.  Heights are kept current: a restructured treelet's interior
// nodes get heights (and sizes) from the merge, and every processed node
// recomputes its own from its final children.
//
// Each treelet is handled by 32 lanes (half a wave64), so the reference's
// warp-32 reductions -- whose tie-breaking depends on the shuffle tree -- are
// reproduced exactly: findLeafToExpand over 2+i lanes and findMinimumDistance
// (per-lane strided minimum over 32 lanes, then a 32-lane tree).  The
// distance matrix lives in LDS; the treelet leaves live in the lanes'
// registers while it is formed and in LDS while it is merged.
#include <algorithm>
#include <vector>

#include "hx_device.h"
#include "hx_internal.h"

namespace hx {

namespace {

constexpr int kG = 32;                         // lanes per treelet
constexpr int kAtrBlock = 256;                 // 8 treelets per workgroup
constexpr int kGroups = kAtrBlock / kG;
constexpr int kMaxT = 30;
constexpr int kTrm = kMaxT * (kMaxT - 1) / 2;  // 435 pairs

constexpr int kBlock = 256;
constexpr int kItems = 16;
constexpr int kTile = kBlock * kItems;

inline unsigned grid_for(int64_t n, int block) { return (unsigned)((n + block - 1) / block); }

// Lower-triangular matrix without its diagonal (TRBuilderUtil.h:44-49,
// ATRBuilderKernels.cu:11-20; the row comes from a float square root, as in
// the reference).
HX_DEV int trm_index(int row, int col) { return ((row - 1) * row) / 2 + col; }
// (row << 8 | col) of an index below kTrm.  sqrt(8 index + 2) lies at least
// 0.008 above 2 row - 1 and 0.05 below 2 row + 1 there, so the hardware's square root
// (1 ulp) gives the same row as the correctly rounded one.
HX_DEV int trm_row_col(int index) {
    const int row = (int)(0.5f * __builtin_amdgcn_sqrtf(8.0f * (float)index + 2.0f) - 0.5f) + 1;
    return row << 8 | (index - (row * (row - 1)) / 2);
}

// TRBuilderUtil.h:100-130 (x*y + x*z + y*z, no validity test).
HX_DEV float atr_area3(float3 mn, float3 mx) {
    const float x = mx.x - mn.x, y = mx.y - mn.y, z = mx.z - mn.z;
    return 2.0f * (x * y + x * z + y * z);
}
HX_DEV float atr_union_area(float3 amn, float3 amx, float3 bmn, float3 bmx) {
    const float x = fmaxf(amx.x, bmx.x) - fminf(amn.x, bmn.x);
    const float y = fmaxf(amx.y, bmx.y) - fminf(amn.y, bmn.y);
    const float z = fmaxf(amx.z, bmx.z) - fminf(amn.z, bmn.z);
    return 2.0f * (x * y + x * z + y * z);
}

template <class T>
HX_DEV T gshfl(T v, int src) { return __shfl(v, src, kG); }
template <class T>
HX_DEV T gshfl_down(T v, int d) { return __shfl_down(v, d, kG); }

// Orders this wave's LDS accesses (no instruction: the wave runs in lockstep).
HX_DEV void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// Maximum over the 32 lanes of a group, in every lane, in VALU moves: rotations
// inside the rows of 16 lanes, then a swap of the two rows.
constexpr int kDppRowRor1 = 0x121, kDppRowRor2 = 0x122, kDppRowRor4 = 0x124, kDppRowRor8 = 0x128;
HX_DEV float group_max(float v) {
    v = fmaxf(v, dpp_move<kDppRowRor8, 0xF>(v));
    v = fmaxf(v, dpp_move<kDppRowRor4, 0xF>(v));
    v = fmaxf(v, dpp_move<kDppRowRor2, 0xF>(v));
    v = fmaxf(v, dpp_move<kDppRowRor1, 0xF>(v));
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    return fmaxf(__int_as_float((int)rows[0]), __int_as_float((int)rows[1]));
}

// v of lane `lane0` of the wave's first group to its lanes and of lane `lane1`
// of the wave to the second group's.
HX_DEV int group_pick(int v, int lane0, int lane1) {
    const int v0 = __builtin_amdgcn_readlane(v, lane0), v1 = __builtin_amdgcn_readlane(v, lane1);
    return lane_id() < kG ? v0 : v1;
}

// Lane of each group's largest value if no group of the wave has a tie or a
// NaN: then every order of comparisons finds the same one.  Otherwise false,
// and the caller takes the reference's shuffle tree, which decides ties.
// `in`: the lane takes part.
HX_DEV bool group_argmax(float v, bool in, int& lane0, int& lane1) {
    const float top = group_max(in ? v : -__builtin_inff());
    const uint64_t nan = ballot64(in && v != v), eq = ballot64(in && v == top);
    const uint32_t lo = (uint32_t)eq, hi = (uint32_t)(eq >> 32);
    lane0 = lo ? __builtin_ctz(lo) : 0;
    lane1 = kG + (hi ? __builtin_ctz(hi) : 0);
    return nan == 0 && (lo & (lo - 1)) == 0 && (hi & (hi - 1)) == 0;
}

// Counts a kept treelet.  Adds to one address are served one after another
// (about 10 ns each), which bound the full heights: 52k treelets took 186 us with
// one counter and take 88 us with 256 on lines of their own.
HX_DEV void count_kept(const AtrArgs& a) {
    const unsigned k = (blockIdx.x * blockDim.x + threadIdx.x) / kG % kAtrCounters;
    atomicAdd(a.accepted + k * kAtrCounterStride, 1);
}

HX_DEV int4 child_record(int l, int r, float al, float ar) {
    return make_int4(l, r, __float_as_int(al), __float_as_int(ar));
}

// formTreelet (TRBuilderUtil.h:171-226): expand the treelet leaf of largest
// area that is an internal node, t-2 times.  Lane i < t ends with treelet leaf
// i in tl, lane i < t-1 with the treelet's internal node i in inode (lane 0:
// the root X, whose record is root).  The steps are a chain of dependent reads;
// a node's record holds its children and their areas, so a step is one read.
HX_DEV void form_treelet(const AtrArgs& a, int X, int4 root, int t, int lane, int& tl, int& inode) {
    const int n = (int)a.n;
    tl = -1;
    inode = -1;
    float tl_area = 0.0f;
    if (lane == 0) {
        tl = root.x;
        tl_area = __int_as_float(root.z);
        inode = X;
    }
    if (lane == 1) {
        tl = root.y;
        tl_area = __int_as_float(root.w);
    }
    for (int it = 0; it < t - 2; ++it) {
        float val = (tl >= n - 1) ? -kMaxFloat : tl_area;
        int e, rep, e0, e1;
        if (group_argmax(val, lane < 2 + it, e0, e1)) {
            e = (lane_id() < kG ? e0 : e1) & (kG - 1);
            rep = group_pick(tl, e0, e1);
        } else {
            int idx = lane;
            for (int k = 2 + it; k > 1; k = (k + 1) / 2) {  // findLeafToExpand
                const int s = k / 2;
                const int oi = gshfl_down(idx, s);
                const float ov = gshfl_down(val, s);
                if (ov > val) {
                    val = ov;
                    idx = oi;
                }
            }
            e = gshfl(idx, 0);
            rep = gshfl(tl, e);
        }
        const int4 rec = a.children[rep];
        if (lane == it + 1) inode = rep;
        if (lane == e) {
            tl = rec.x;
            tl_area = __int_as_float(rec.z);
        }
        if (lane == it + 2) {
            tl = rec.y;
            tl_area = __int_as_float(rec.w);
        }
    }
}

// LDS of one 32-lane group: the distance matrix and the state of the rows
// (box, cost, node, size, height), read by every lane as broadcasts.
struct AtrGroup {
    float4 lo[kG];  // box minimum, SAH cost
    float4 hi[kG];  // box maximum, node
    int2 rh[kG];    // references, height
    float d[kTrm + 1];
};

// The treelet of X by 32 lanes.  A wave holds two treelets and the levels of
// the upper tree have fewer treelets than the chip has waves, so a level takes
// what one treelet takes, a serial chain of t - 2 expansions and t - 1 joins
// (9 leaves: 3.5 + 6.2 us of a 14 us level).  So a join is short: the minimum
// by row rotations, ties alone by the reference's tree; the rows' state in LDS,
// read as broadcasts together; no square root to the last bit.  1M triangles:
// the 66 levels of a build took 1941 us; 34 of them and the two launches of
// k_atr_top now take 1241 us (count_kept included).
HX_DEV void atr_treelet(const AtrArgs& a, int X, int lane, AtrGroup& g) {
    const int n = (int)a.n;
    const int t = a.treelet_size;
    float* const D = g.d;

    // The climb step at X (ATRBuilderKernels.cu:293-310): children are final.
    const int4 root = a.children[X];
    const int xl = root.x, xr = root.y;
    const float costX = a.ct * a.area[X] + a.cost[xl] + a.cost[xr];
    const int hl = xl >= n - 1 ? 0 : a.height[xl];
    const int hr = xr >= n - 1 ? 0 : a.height[xr];
    const int heightX = 1 + max(hl, hr);

    int tl, inode;
    form_treelet(a, X, root, t, lane, tl, inode);

    // Treelet leaves: node, box, cost, size, height per lane.
    int node = tl, rnode = -1, mrefs = 0, mh = 0;
    float mcost = 0.0f, larea = 0.0f, rarea = 0.0f;
    float3 mn = make_float3(0.0f, 0.0f, 0.0f), mx = mn;
    if (lane < t) {
        const float4 bmn = a.nmin[tl], bmx = a.nmax[tl];
        const float sah = a.cost[tl];
        int refs = 1, hgt = 0;
        if (tl < n - 1) {
            refs = a.refs[tl];
            hgt = a.height[tl];
        }
        mn = make_float3(bmn.x, bmn.y, bmn.z);
        mx = make_float3(bmx.x, bmx.y, bmx.z);
        g.lo[lane] = make_float4(mn.x, mn.y, mn.z, sah);
        g.hi[lane] = make_float4(mx.x, mx.y, mx.z, __int_as_float(tl));
        g.rh[lane] = make_int2(refs, hgt);
    }
    wave_lds_fence();

    // calculateDistancesMatrix (ATRBuilderKernels.cu:22-64): every pair.
    const int pairs = t * (t - 1) / 2;
    for (int e = lane; e < pairs; e += kG) {
        const int rc = trm_row_col(e), row = rc >> 8, col = rc & 0xFF;
        D[e] = atr_union_area(xyz(g.lo[row]), xyz(g.hi[row]), xyz(g.lo[col]), xyz(g.hi[col]));
    }
    wave_lds_fence();

    for (int lastRow = t - 1; lastRow > 0; --lastRow) {
        // What does not hang on the join is read first.
        const float dLast = D[trm_index(lastRow, min(lane, lastRow - 1))];
        const float4 lastLo = g.lo[lastRow], lastHi = g.hi[lastRow];
        const int2 lastRh = g.rh[lastRow];
        const int newId = group_pick(inode, lastRow - 1, kG + lastRow - 1);
        // findMinimumDistance (:81-94): strided minimum, then a 32-lane tree.
        const int msize = lastRow * (lastRow + 1) / 2;
        int mi = 0;
        float md = kMaxFloat;
        for (int j = lane; j < msize; j += kG) {
            const float d = D[j];
            if (d < md) {
                md = d;
                mi = j;
            }
        }
        int e0, e1;
        if (group_argmax(-md, true, e0, e1)) {
            mi = group_pick(mi, e0, e1);
        } else {
            for (int s = kG / 2; s >= 1; s >>= 1) {
                const int oi = gshfl_down(mi, s);
                const float od = gshfl_down(md, s);
                if (od < md) {
                    md = od;
                    mi = oi;
                }
            }
            mi = gshfl(mi, 0);
        }
        const int join = trm_row_col(mi), joinCol = join & 0xFF, joinRow = join >> 8;

        // updateState (:96-158): the merged node takes row joinCol, row
        // lastRow moves to joinRow.
        const float4 rLo = g.lo[joinRow], rHi = g.hi[joinRow], cLo = g.lo[joinCol], cHi = g.hi[joinCol];
        const int2 rRh = g.rh[joinRow], cRh = g.rh[joinCol];
        const float ssum = rLo.w + cLo.w;
        const float la = atr_area3(xyz(rLo), xyz(rHi)), ra = atr_area3(xyz(cLo), xyz(cHi));
        const float3 amn = make_float3(fminf(cLo.x, rLo.x), fminf(cLo.y, rLo.y), fminf(cLo.z, rLo.z));
        const float3 amx = make_float3(fmaxf(cHi.x, rHi.x), fmaxf(cHi.y, rHi.y), fmaxf(cHi.z, rHi.z));
        const int refsNew = rRh.x + cRh.x;
        const int hNew = 1 + max(rRh.y, cRh.y);
        const float c = ssum + a.ct * atr_area3(amn, amx);
        if (lane == lastRow) {
            node = __float_as_int(rHi.w);
            rnode = __float_as_int(cHi.w);
            larea = la;
            rarea = ra;
            mcost = c;
            mrefs = refsNew;
            mh = hNew;
        }
        const bool isCol = lane == joinCol;
        if (lane == joinRow) {
            mn = xyz(lastLo);
            mx = xyz(lastHi);
        }
        if (isCol || lane == lastRow) {
            mn = amn;
            mx = amx;
        }

        if (lastRow > 1) {
            if (isCol || lane == joinRow) {
                g.lo[lane] = isCol ? make_float4(amn.x, amn.y, amn.z, c) : lastLo;
                g.hi[lane] = isCol ? make_float4(amx.x, amx.y, amx.z, __int_as_float(newId)) : lastHi;
                g.rh[lane] = isCol ? make_int2(refsNew, hNew) : lastRh;
            }
            // updateDistancesMatrix (:160-196): row lastRow moves to joinRow,
            // then row/column joinCol is recomputed from the merged box (a
            // union's area does not depend on the order of its two boxes).
            if (lane < lastRow && lane != joinRow) D[trm_index(max(joinRow, lane), min(joinRow, lane))] = dLast;
            wave_lds_fence();
            if (lane < lastRow && lane != joinCol)
                D[trm_index(max(joinCol, lane), min(joinCol, lane))] = atr_union_area(mn, mx, amn, amx);
            wave_lds_fence();
        }
    }

    // updateTreelet (:198-228): keep the new treelet if its cost is lower.
    const float newCost = gshfl(mcost, 1);
    const int vid = gshfl(inode, lane >= 1 ? lane - 1 : 0);
    if (newCost < costX) {
        if (lane >= 1 && lane < t) {
            a.left[vid] = node;
            a.right[vid] = rnode;
            a.children[vid] = child_record(node, rnode, larea, rarea);
            a.parent[node] = vid;
            a.parent[rnode] = vid;
            a.cost[vid] = mcost;
            a.nmin[vid] = make_float4(mn.x, mn.y, mn.z, 0.0f);
            a.nmax[vid] = make_float4(mx.x, mx.y, mx.z, 0.0f);
            a.area[vid] = atr_area3(mn, mx);
            a.refs[vid] = mrefs;
            a.height[vid] = mh;
        }
        if (lane == 0) count_kept(a);
    } else if (lane == 0) {
        a.cost[X] = costX;
        a.height[X] = heightX;
    }
}

// The cost climb step for a node that is not restructured (ATRBuilderKernels.cu
// :293-310): every iteration recomputes it, which matters for interior nodes a
// kept treelet gave a cost in merge order.
HX_DEV void atr_climb_cost(const AtrArgs& a, int v) {
    a.cost[v] = a.ct * a.area[v] + a.cost[a.left[v]] + a.cost[a.right[v]];
}

// One treelet per 32-lane group; task = index into the height bucket.
__global__ __launch_bounds__(kAtrBlock) void k_atr_level(AtrArgs a, const int32_t* __restrict__ list, int count) {
    __shared__ AtrGroup s_group[kGroups];
    const int grp = threadIdx.x / kG;
    const int task = blockIdx.x * kGroups + grp;
    if (task >= count) return;  // whole 32-lane groups leave together
    atr_treelet(a, list[task], threadIdx.x & (kG - 1), s_group[grp]);
}

// The remaining heights, none with more than kTopTasks nodes in a bucket, by
// one workgroup: what a height wrote is in this CU's cache when the next one
// reads it, and there are no launches between them.  A height takes 12 us here and 14 us
// as a launch of its own.
constexpr int kTopThreads = 1024;
constexpr int kTopTasks = 64;
__global__ __launch_bounds__(kTopThreads) void k_atr_top(AtrArgs a, int bucket, int buckets, int offset, bool costs) {
    constexpr int G = kTopThreads / kG;
    __shared__ AtrGroup s_group[G];
    const int grp = threadIdx.x / kG;
    for (int b = bucket; b < buckets; ++b) {
        const int count = a.hist[b];
        if (count == 0) continue;
        const int32_t* list = a.list + offset;
        if (b & 1) {
            for (int k = grp; k < count; k += G) atr_treelet(a, list[k], threadIdx.x & (kG - 1), s_group[grp]);
        } else if (costs) {
            for (int k = threadIdx.x; k < count; k += kTopThreads) atr_climb_cost(a, list[k]);
        }
        offset += count;
        __syncthreads();  // this height's nodes before the next one's reads
    }
}

// The records of form_treelet, from the prepared hierarchy.
__global__ __launch_bounds__(kBlock) void k_atr_children(AtrArgs a) {
    const int v = blockIdx.x * kBlock + threadIdx.x;
    if (v >= (int)a.n - 1) return;
    const int l = a.left[v], r = a.right[v];
    a.children[v] = child_record(l, r, a.area[l], a.area[r]);
}

__global__ __launch_bounds__(kBlock) void k_atr_small(AtrArgs a, const int32_t* __restrict__ list, int count) {
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    atr_climb_cost(a, list[k]);
}

// ---- TR: optimal treelet restructuring (TRBuilderKernels.cu:11-476) ----
//
// The treelet has 7 leaves (TRBuilder::setTreeletSize accepts 7 only) and is
// formed as ATRBVH's.  Its 128 leaf subsets get their union areas, the leaves
// their current costs, and a DP over the subsets by size gives every subset's
// optimal cost C(S) = min(ct A(S) + min_P [C(P) + C(S\P)], ci A(S) R), R the
// root's reference count.  The partitions are enumerated as the reference
// does, so every split leaves the subset's lowest leaf on the right and ties
// go as there: subsets of 2..5 leaves scan their partitions in one lane
// (first strict minimum), the 6-leaf subsets split theirs over 4 lanes and the
// whole treelet over 32, each reduced by the reference's shuffle-down tree.
constexpr int kTrT = 7;
constexpr int kTrS = 1 << kTrT;

struct TrSchedule {
    uint8_t subset[112];  // subsets of 2..5 leaves, grouped by size
    uint8_t off[5];       // group of size 2 + i: [off[i], off[i+1])
};
constexpr int tr_popc(int v) {
    int c = 0;
    for (; v; v >>= 1) c += v & 1;
    return c;
}
constexpr TrSchedule make_tr_schedule() {
    TrSchedule r{};
    int k = 0;
    for (int size = 2; size <= kTrT - 2; ++size) {
        r.off[size - 2] = (uint8_t)k;
        for (int v = 1; v < kTrS; ++v)
            if (tr_popc(v) == size) r.subset[k++] = (uint8_t)v;
    }
    r.off[kTrT - 3] = (uint8_t)k;
    return r;
}
static_assert(make_tr_schedule().off[4] == 112, "subsets of 2..5 of 7 leaves");
__constant__ TrSchedule kTrSchedule = make_tr_schedule();

// processSchedule's per-subset step (TRBuilderKernels.cu:96-116).
HX_DEV void tr_finish(float* C, uint8_t* M, int s, float opt, int best, float ct, float ci, float R) {
    const float A = C[s];
    C[s] = fminf(ct * A + opt, ci * A * R);
    M[s] = (uint8_t)best;
}

// reduceOptimal (TRBuilderKernels.cu:11-20): shuffle down by values/2 ... 1,
// a lane keeps its own pair unless the other is strictly cheaper.
HX_DEV void tr_reduce(float& opt, int& best, int values) {
    for (int d = values >> 1; d > 0; d >>= 1) {
        const float ov = gshfl_down(opt, d);
        const int ob = gshfl_down(best, d);
        if (ov < opt) {
            opt = ov;
            best = ob;
        }
    }
}

// One treelet per 32-lane group; task = index into the height bucket.
__global__ __launch_bounds__(kAtrBlock) void k_tr_level(AtrArgs a, const int32_t* __restrict__ list, int count) {
    __shared__ float s_cost[kGroups][kTrS];
    __shared__ uint8_t s_mask[kGroups][kTrS];
    __shared__ float s_box[kGroups][kTrT][6];
    __shared__ int s_leaf[kGroups][3][kTrT];       // node, references, height
    __shared__ int s_inode[kGroups][kTrT - 1];
    __shared__ int s_rec[kGroups][6][kTrT - 1];    // node, mask, left, right, cost subset, height
    __shared__ int s_nrec[kGroups];
    const int grp = threadIdx.x / kG;
    const int lane = threadIdx.x & (kG - 1);
    const int task = blockIdx.x * kGroups + grp;
    if (task >= count) return;  // whole 32-lane groups leave together
    float* C = s_cost[grp];
    uint8_t* M = s_mask[grp];
    const int n = (int)a.n;
    const int X = list[task];
    const float ct = a.ct, ci = a.ci;

    // The climb step at X (TRBuilderKernels.cu:391-407): children are final.
    const int4 root = a.children[X];
    const int xl = root.x, xr = root.y;
    const float costX = ct * a.area[X] + a.cost[xl] + a.cost[xr];
    const int hl = xl >= n - 1 ? 0 : a.height[xl];
    const int hr = xr >= n - 1 ? 0 : a.height[xr];
    const int heightX = 1 + max(hl, hr);
    const float R = (float)a.refs[X];

    int tl, inode;
    form_treelet(a, X, root, kTrT, lane, tl, inode);
    float leafCost = 0.0f;
    if (lane < kTrT) {
        const float4 bmn = a.nmin[tl], bmx = a.nmax[tl];
        float* b = s_box[grp][lane];
        b[0] = bmn.x;
        b[1] = bmn.y;
        b[2] = bmn.z;
        b[3] = bmx.x;
        b[4] = bmx.y;
        b[5] = bmx.z;
        s_leaf[grp][0][lane] = tl;
        s_leaf[grp][1][lane] = tl < n - 1 ? a.refs[tl] : 1;
        s_leaf[grp][2][lane] = tl < n - 1 ? a.height[tl] : 0;
        leafCost = a.cost[tl];
    }
    if (lane < kTrT - 1) s_inode[grp][lane] = inode;
    wave_lds_fence();

    // calculateSubsetSurfaceAreas (:22-81): lane l owns subsets 4l .. 4l+3;
    // unions are exact, so their order is free.
    for (int j = 0; j < kTrS / kG; ++j) {
        const int v = (kTrS / kG) * lane + j;
        float3 mn = make_float3(kMaxFloat, kMaxFloat, kMaxFloat);
        float3 mx = make_float3(-kMaxFloat, -kMaxFloat, -kMaxFloat);
        for (int i = 0; i < kTrT; ++i) {
            if (v >> i & 1) {
                const float* b = s_box[grp][i];
                mn = make_float3(fminf(b[0], mn.x), fminf(b[1], mn.y), fminf(b[2], mn.z));
                mx = make_float3(fmaxf(b[3], mx.x), fmaxf(b[4], mx.y), fmaxf(b[5], mx.z));
            }
        }
        C[v] = atr_area3(mn, mx);
    }
    wave_lds_fence();
    if (lane < kTrT) C[1 << lane] = leafCost;  // :433-437
    wave_lds_fence();

    // processSchedule (:84-114): subsets of 2..5 leaves, one size at a time.
#pragma unroll
    for (int g = 0; g < kTrT - 3; ++g) {
        for (int k = kTrSchedule.off[g] + lane; k < kTrSchedule.off[g + 1]; k += kG) {
            const int v = kTrSchedule.subset[k];
            float opt = kMaxFloat;
            int best = 0;
            const int delta = (v - 1) & v;
            int p = (-delta) & v;
            while (p != 0) {
                const float c = C[p] + C[p ^ v];
                if (c < opt) {
                    opt = c;
                    best = p;
                }
                p = (p - delta) & v;
            }
            tr_finish(C, M, v, opt, best, ct, ci, R);
        }
        wave_lds_fence();
    }

    // processSubsets (:116-196): the 7 subsets of 6 leaves over 4 lanes each.
    {
        float opt = kMaxFloat;
        int best = 0;
        const int g = lane >> 2;
        const int v = (kTrS - 1) & ~(1 << g);
        if (lane < 4 * kTrT) {
            const int leftMask = -(1 << max(g - 1, 0));
            int base = (lane & 3) + 1;
            int p = (((base & leftMask) << 1) | (base & ~leftMask)) << 1;
            for (int j = lane & 3; j < (1 << (kTrT - 2)) - 1; j += 4) {
                const float c = C[p] + C[p ^ v];
                if (c < opt) {
                    opt = c;
                    best = p;
                }
                base += 4;
                p = (((base & leftMask) << 1) | (base & ~leftMask)) << 1;
            }
        }
        tr_reduce(opt, best, 4);
        if (lane < 4 * kTrT && (lane & 3) == 0) tr_finish(C, M, v, opt, best, ct, ci, R);
    }
    wave_lds_fence();
    {
        float opt = kMaxFloat;
        int best = 0;
        int p = (lane + 1) * 2;
        for (int j = lane; j < (1 << (kTrT - 1)) - 1; j += kG) {
            const float c = C[p] + C[p ^ (kTrS - 1)];
            if (c < opt) {
                opt = c;
                best = p;
            }
            p += 2 * kG;
        }
        tr_reduce(opt, best, kG);
        if (lane == 0) tr_finish(C, M, kTrS - 1, opt, best, ct, ci, R);
    }
    wave_lds_fence();

    // updateTreelet (:198-324): keep the optimal tree if it is cheaper.  Lane 0
    // lays it out as the reference's stack rounds do: per round, the left
    // sides of the stacked nodes take the next internal nodes in stack order,
    // then the right sides; new internal nodes are stacked in that order.
    const bool keep = C[kTrS - 1] < costX;
    int(*rec)[kTrT - 1] = s_rec[grp];  // rec[field][record]
    if (keep && lane == 0) {
        const int* leafNode = s_leaf[grp][0];
        const int* leafH = s_leaf[grp][2];
        int nrec = 1, next = 1, rb = 0;
        rec[0][0] = X;
        rec[1][0] = kTrS - 1;
        rec[4][0] = 0;
        while (rb < nrec) {
            const int re = nrec;
            for (int side = 0; side < 2; ++side) {
                for (int i = rb; i < re; ++i) {
                    const int part = M[rec[1][i]];
                    const int v = side == 0 ? part : (part ^ rec[1][i]);
                    int child;
                    // A finite kept cost gives every subset on the tree a
                    // split; the bounds only keep non-finite boxes in range.
                    if (__popc(v) > 1 && nrec < kTrT - 1) {
                        child = s_inode[grp][next++];
                        rec[0][nrec] = child;
                        rec[1][nrec] = v;
                        rec[4][nrec] = part;  // the reference's costs[partition], both sides
                        ++nrec;
                    } else {
                        child = leafNode[max(__ffs(v) - 1, 0)];
                    }
                    rec[2 + side][i] = child;
                }
            }
            rb = re;
        }
        s_nrec[grp] = nrec;
        // Heights bottom-up: every record's children come after it.
        for (int i = nrec - 1; i >= 0; --i) {
            const int part = M[rec[1][i]];
            int h[2];
            for (int side = 0; side < 2; ++side) {
                const int v = side == 0 ? part : (part ^ rec[1][i]);
                int hv = 0;
                if (__popc(v) > 1) {
                    for (int k = i + 1; k < nrec; ++k)
                        if (rec[1][k] == v) hv = rec[5][k];
                } else {
                    hv = leafH[max(__ffs(v) - 1, 0)];
                }
                h[side] = hv;
            }
            rec[5][i] = 1 + max(h[0], h[1]);
        }
    }
    wave_lds_fence();
    if (keep && lane < s_nrec[grp]) {
        const int node = rec[0][lane], v = rec[1][lane], l = rec[2][lane], r = rec[3][lane];
        a.left[node] = l;
        a.right[node] = r;
        a.parent[l] = node;
        a.parent[r] = node;
        int refs = 0;
        for (int i = 0; i < kTrT; ++i)
            if (v >> i & 1) refs += s_leaf[grp][1][i];
        // Box of a set of treelet leaves; a child's record area is the area
        // that its own lane stores.
        auto box_of = [&](int set, float3& mn, float3& mx) {
            mn = make_float3(kMaxFloat, kMaxFloat, kMaxFloat);
            mx = make_float3(-kMaxFloat, -kMaxFloat, -kMaxFloat);
            for (int i = 0; i < kTrT; ++i) {
                if (set >> i & 1) {
                    const float* b = s_box[grp][i];
                    mn = make_float3(fminf(b[0], mn.x), fminf(b[1], mn.y), fminf(b[2], mn.z));
                    mx = make_float3(fmaxf(b[3], mx.x), fmaxf(b[4], mx.y), fmaxf(b[5], mx.z));
                }
            }
        };
        float3 mn, mx;
        box_of(M[v], mn, mx);
        const float larea = atr_area3(mn, mx);
        box_of(M[v] ^ v, mn, mx);
        a.children[node] = child_record(l, r, larea, atr_area3(mn, mx));
        box_of(v, mn, mx);
        a.refs[node] = refs;
        a.height[node] = rec[5][lane];
        if (lane > 0) {  // the root keeps its box and its climb cost
            a.nmin[node] = make_float4(mn.x, mn.y, mn.z, 0.0f);
            a.nmax[node] = make_float4(mx.x, mx.y, mx.z, 0.0f);
            a.area[node] = atr_area3(mn, mx);
            a.cost[node] = C[rec[4][lane]];
        }
    }
    if (lane == 0) {
        a.cost[X] = costX;
        if (keep) count_kept(a);
        else a.height[X] = heightX;
    }
}

// Bucket of an internal node: 2 * height + (references >= gamma).
constexpr int kBuckets = 2 * kAtrMaxLevels;

HX_DEV int bucket_of(const int32_t* refs, const int32_t* height, int v, int gamma) {
    return min(2 * height[v] + (refs[v] >= gamma ? 1 : 0), kBuckets);
}

// Bucket counts: per-tile LDS counts, then one global add per (tile, bucket).
__global__ __launch_bounds__(kBlock) void k_atr_count(const int32_t* __restrict__ refs,
                                                      const int32_t* __restrict__ height, int m, int gamma,
                                                      int32_t* __restrict__ hist) {
    __shared__ int s_cnt[kBuckets + 1];
    for (int i = threadIdx.x; i <= kBuckets; i += kBlock) s_cnt[i] = 0;
    __syncthreads();
    const int64_t base = blockIdx.x * (int64_t)kTile;
    for (int k = 0; k < kItems; ++k) {
        const int64_t v = base + k * kBlock + threadIdx.x;
        if (v < m) atomicAdd(&s_cnt[bucket_of(refs, height, (int)v, gamma)], 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i <= kBuckets; i += kBlock)
        if (s_cnt[i]) atomicAdd(&hist[i], s_cnt[i]);
}

// Scatter into the buckets (order inside a bucket is free: its nodes are
// independent).  cursor[h] starts at the bucket's offset.
__global__ __launch_bounds__(kBlock) void k_atr_scatter(const int32_t* __restrict__ refs,
                                                        const int32_t* __restrict__ height, int m, int gamma,
                                                        int32_t* __restrict__ cursor, int32_t* __restrict__ list) {
    __shared__ int s_cnt[kBuckets];
    __shared__ int s_base[kBuckets];
    for (int i = threadIdx.x; i < kBuckets; i += kBlock) s_cnt[i] = 0;
    __syncthreads();
    const int64_t base = blockIdx.x * (int64_t)kTile;
    int lvl[kItems], loc[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int64_t v = base + k * kBlock + threadIdx.x;
        lvl[k] = -1;
        if (v < m) {
            lvl[k] = bucket_of(refs, height, (int)v, gamma);
            loc[k] = atomicAdd(&s_cnt[lvl[k]], 1);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kBuckets; i += kBlock)
        if (s_cnt[i]) s_base[i] = atomicAdd(&cursor[i], s_cnt[i]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if (lvl[k] >= 0) list[s_base[lvl[k]] + loc[k]] = (int)(base + k * kBlock + threadIdx.x);
}

// Sum of the counters into the first one.
__global__ __launch_bounds__(kAtrCounters) void k_atr_kept(int32_t* __restrict__ accepted) {
    static_assert(kAtrCounters == 256, "four waves");
    __shared__ int s_sum[kAtrCounters / kWave];
    const int v = wave_sum_i32(accepted[threadIdx.x * kAtrCounterStride]);
    if (lane_id() == 0) s_sum[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) accepted[0] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

__global__ void k_atr_zero(int32_t* __restrict__ p, int count) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) p[i] = 0;
}

// Buckets the internal nodes by (height, >= gamma references); returns the
// per-bucket counts on the host and leaves the nodes in a.list.
int bucket_by_height(Context* c, const AtrArgs& a, int gamma, std::vector<int>& counts) {
    const int m = (int)a.n - 1;
    hipLaunchKernelGGL(k_atr_zero, dim3(4), dim3(kBlock), 0, c->stream, a.hist, kBuckets + 1);
    HX_TRY(check_launch("atr_zero"));
    const unsigned tiles = grid_for(m, kTile);
    hipLaunchKernelGGL(k_atr_count, dim3(tiles), dim3(kBlock), 0, c->stream, a.refs, a.height, m, gamma, a.hist);
    HX_TRY(check_launch("atr_count"));
    counts.assign(kBuckets + 1, 0);
    HX_HIP(hipMemcpyAsync(counts.data(), a.hist, sizeof(int) * (kBuckets + 1), hipMemcpyDeviceToHost, c->stream));
    HX_HIP(hipStreamSynchronize(c->stream));
    if (counts[kBuckets] != 0) {
        set_error("a subtree is deeper than %d levels", kAtrMaxLevels - 1);
        return HX_ERR_UNSUPPORTED;
    }
    std::vector<int> offs(kBuckets, 0);
    int run = 0;
    for (int b = 0; b < kBuckets; ++b) {
        offs[b] = run;
        run += counts[b];
    }
    HX_HIP(hipMemcpyAsync(a.cursor, offs.data(), sizeof(int) * kBuckets, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_atr_scatter, dim3(tiles), dim3(kBlock), 0, c->stream, a.refs, a.height, m, gamma,
                       a.cursor, a.list);
    HX_TRY(check_launch("atr_scatter"));
    // The host vector must outlive the asynchronous upload.
    HX_HIP(hipStreamSynchronize(c->stream));
    return HX_OK;
}

}  // namespace

int launch_relabel_by_height(Context* c, const AtrArgs& a, const PlocArgs& relabel) {
    // Depth-first relabelling, parents first: buckets by height, top down.
    LaunchScope ls(c, "relabel");
    std::vector<int> counts;
    HX_TRY(bucket_by_height(c, a, 0, counts));
    HX_HIP(hipMemcpyAsync(relabel.last, a.refs, sizeof(int32_t) * (size_t)(a.n - 1), hipMemcpyDeviceToDevice,
                          c->stream));
    std::vector<int> offs(kBuckets + 1, 0);
    for (int b = 0; b < kBuckets; ++b) offs[b + 1] = offs[b] + counts[b];
    // Both buckets of a height are contiguous: one step per height.
    std::vector<int2> segs;
    for (int h = kAtrMaxLevels - 1; h >= 0; --h) {
        const int cnt = counts[2 * h] + counts[2 * h + 1];
        if (cnt > 0) segs.push_back(make_int2(offs[2 * h], cnt));
    }
    return launch_tree_down_steps(c, relabel, a.list, segs);
}

namespace {

// ATRBuilder::optimize (ATRBuilder.cpp:80-177) and TRBuilder::optimize
// (TRBuilder.cpp:140-191) share the loop: gamma starts at the treelet size and
// doubles per iteration, stopping once it exceeds the reference count.
int launch_treelets(Context* c, const AtrArgs& a, const PlocArgs& relabel, int64_t* accepted_out, bool tr) {
    const int64_t n = a.n;
    hipLaunchKernelGGL(k_atr_zero, dim3(8), dim3(kBlock), 0, c->stream, a.accepted, kAtrCounters * kAtrCounterStride);
    HX_TRY(check_launch("atr_zero"));
    if (n > 1 && a.iterations > 0) {
        hipLaunchKernelGGL(k_atr_children, dim3(grid_for(n - 1, kBlock)), dim3(kBlock), 0, c->stream, a);
        HX_TRY(check_launch("atr_children"));
    }
    std::vector<int> counts;
    int64_t gamma = a.treelet_size;
    {
        LaunchScope ls(c, tr ? "tr_optimize" : "atr_optimize");
        for (int i = 0; i < a.iterations; ++i) {
            HX_TRY(bucket_by_height(c, a, (int)std::min<int64_t>(gamma, INT32_MAX), counts));
            int buckets = kBuckets;
            while (buckets > 0 && counts[buckets - 1] == 0) --buckets;
            int top = buckets;  // first bucket of k_atr_top
            if (!tr)
                while (top > 0 && counts[top - 1] <= kTopTasks) --top;
            int off = 0;
            for (int b = 0; b < buckets; ++b) {
                const int cnt = counts[b];
                if (b == top) {
                    hipLaunchKernelGGL(k_atr_top, dim3(1), dim3(kTopThreads), 0, c->stream, a, top, buckets, off,
                                       i > 0);
                    HX_TRY(check_launch("atr_top"));
                    break;
                }
                if (cnt > 0 && (b & 1)) {
                    if (tr) {
                        hipLaunchKernelGGL(k_tr_level, dim3(grid_for(cnt, kGroups)), dim3(kAtrBlock), 0,
                                           c->stream, a, (const int32_t*)(a.list + off), cnt);
                        HX_TRY(check_launch("tr_level"));
                    } else {
                        hipLaunchKernelGGL(k_atr_level, dim3(grid_for(cnt, kGroups)), dim3(kAtrBlock), 0,
                                           c->stream, a, (const int32_t*)(a.list + off), cnt);
                        HX_TRY(check_launch("atr_level"));
                    }
                } else if (cnt > 0 && i > 0) {
                    // The first iteration's small-node costs are the prepared ones.
                    hipLaunchKernelGGL(k_atr_small, dim3(grid_for(cnt, kBlock)), dim3(kBlock), 0, c->stream, a,
                                       (const int32_t*)(a.list + off), cnt);
                    HX_TRY(check_launch("atr_small"));
                }
                off += cnt;
            }
            gamma *= 2;  // ATRBuilder.cpp:163-171
            if (gamma > n) break;
        }
    }
    HX_TRY(launch_relabel_by_height(c, a, relabel));
    if (accepted_out) {
        hipLaunchKernelGGL(k_atr_kept, dim3(1), dim3(kAtrCounters), 0, c->stream, a.accepted);
        HX_TRY(check_launch("atr_kept"));
        int32_t acc = 0;
        HX_HIP(hipMemcpyAsync(&acc, a.accepted, sizeof(acc), hipMemcpyDeviceToHost, c->stream));
        HX_HIP(hipStreamSynchronize(c->stream));
        *accepted_out = acc;
    }
    return HX_OK;
}

}  // namespace

int launch_atr(Context* c, const AtrArgs& a, const PlocArgs& relabel, int64_t* accepted_out) {
    return launch_treelets(c, a, relabel, accepted_out, false);
}

int launch_tr(Context* c, const AtrArgs& a, const PlocArgs& relabel, int64_t* accepted_out) {
    if (a.treelet_size != kTrT) return HX_ERR_INVALID_ARG;
    return launch_treelets(c, a, relabel, accepted_out, true);
}

}  // namespace hx
