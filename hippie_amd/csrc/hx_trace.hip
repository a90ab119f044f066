// hx_trace.hip -- persistent while-while traversal of the Bin BVH for gfx950,
// plus the Morton ray keys used by the sorted trace.
//
// Reference (src/hippie/): rt/tracer/HipTracerBinKernels.cu:19-286 (trace),
// :572-842 (traceSort), rt/tracer/HipTracerKernels.h:29-199,
// rt/ray/RayBufferKernels.cu:12-56,492-614.
//
// Wave64 design: each wave takes runs of rays for its terminated lanes (64-bit
// ballot + mbcnt) from a pool of its own (RayPool), traverses with the
// Aila-Laine while-while loop, postpones leaves, and refills when fewer than
// fetch_threshold of its lanes are still busy.
#include "hx_device.h"
#include "hx_internal.h"

namespace hx {

namespace {

constexpr int kTraceBlock = 256;
constexpr int kStackSize = 64;                 // HipTracerBinKernels.cu:5
constexpr int32_t kSentinel = 0x76543210;      // HipTracerKernels.h:11

// fminf/fmaxf (v_min_f32 / v_max_f32: a NaN operand yields the other, -0
// orders below +0, as the reference's fminf/fmaxf do) and the integer min/max
// on float bits of HipTracerKernels.h:144-195 (spanBeginKepler / spanEndKepler).
HX_DEV float fmin_s(float a, float b) { return fminf(a, b); }
HX_DEV float fmax_s(float a, float b) { return fmaxf(a, b); }
HX_DEV float span_begin(float a0, float a1, float b0, float b1, float c0, float c1, float d) {
    const int c = max(min(__float_as_int(c0), __float_as_int(c1)), __float_as_int(d));
    return __int_as_float(max(max(__float_as_int(fmin_s(a0, a1)), __float_as_int(fmin_s(b0, b1))), c));
}
HX_DEV float span_end(float a0, float a1, float b0, float b1, float c0, float c1, float d) {
    const int c = min(max(__float_as_int(c0), __float_as_int(c1)), __float_as_int(d));
    return __int_as_float(min(min(__float_as_int(fmax_s(a0, a1)), __float_as_int(fmax_s(b0, b1))), c));
}

// The rays of one wave.  Every wave starts on its own run of rays and, when it
// is used up, takes the next run with one atomicAdd on the launch's counter.
// One atomic on one address per refill is what held traces back before: device
// atomics on an address shared by the eight XCDs serialise at the memory side
// (~10 ns each), and 1,048,576 rays half of which miss at the root take one per
// ~24 rays.  With runs of up to kRunMax rays those rays went from 516 to 419 us
// and 1,000,000 diffuse rays from 900 to 704 us.  Runs shrink with the rays left
// (1 / (4 x waves) of them, at least one ray per lane) so that the last waves
// finish together: a fixed run of 1/2 of a wave's share cost 15 % on 16.7M
// diffuse rays.
// Batched rays keep to runs of 64: the rays in flight belong to few meshes then,
// whose trees the caches hold (67.1M rays into 512 meshes 280 -> 226 ms, 241 with
// a refill at a time; with 1M atomics in that time the counter does not bound it).
//
// Rays from one point (`alike`, see alike_pays) are handed out a refill at a time.
// Neighbours among them cost alike, so a wave that stays on its own run in a
// costly place carries several groups of long-lived rays, each at another depth;
// when all waves take the next rays in turn it carries one such group among short
// ones.  16.7M sorted primaries over as many triangles: 2.93 -> 2.57 G VALU and
// 170 -> 124 M vector-load instructions.
constexpr int kControlAlike = 2;   // word of TraceArgs::control
constexpr int kRunMax = 256, kRunMaxBatch = 64;
struct RayPool {
    int next, end;   // this wave's rays
    int base;        // first ray of the latest run: the rays left start about here
    int dyn0;        // first ray that is handed out by the counter
    int n, lanes, shift, most;
    bool alike;

    HX_DEV int run() const { return max(lanes, min((n - base) >> shift, most)); }
    HX_DEV void start(const TraceArgs& a, bool one_point) {
        n = (int)a.n_rays;
        lanes = a.lanes;
        shift = a.run_shift;
        most = a.ray_mesh ? kRunMaxBatch : kRunMax;
        base = 0;
        alike = one_point;
        const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kTraceBlock / kWave) + threadIdx.x / kWave);
        const int r = alike ? lanes : run();
        next = wave * r;
        end = min(next + r, n);
        dyn0 = base = (int)gridDim.x * (kTraceBlock / kWave) * r;
    }
    // A ray slot for each lane with `want` (>= n: none left); called by the
    // whole wave.  mask, count: the lanes that want one.
    HX_DEV int take(bool want, uint64_t mask, int count, int32_t* counter) {
        const int below = count_below(mask);
        const int avail = max(end - next, 0);
        int mine = next + below;
        if (count > avail) {
            int first = n;
            const int r = alike ? count : run();
            if (base < n) {
                if (want && below == 0) first = atomicAdd(counter, r);
                first = dyn0 + __builtin_amdgcn_readlane(first, __ffsll((unsigned long long)mask) - 1);
            }
            if (below >= avail) mine = first + (below - avail);
            base = first;
            next = first + (count - avail);
            end = min(first + r, n);
        } else {
            next += count;
        }
        return mine;
    }
};

// SGPR budget of the trace kernels.  Above 80 scalar registers (96 with the
// 16 the trap handler keeps) a SIMD holds 7 waves instead of 8 although the
// occupancy query still says 8: 16.7M diffuse rays took 7.25 ms with 82 to 94
// registers and 6.27 ms with 76 to 80.  The Bin kernel is held to the 64 vector
// registers of 8 waves too (it needs 64 or 65).
#define HX_TRACE_KERNEL __global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_num_sgpr(80)))

// Traversal stack: entries [0, LDS_DEPTH) in LDS, one column per lane (entry e
// of lane t at e * kTraceBlock + t, so a wave's accesses hit distinct banks);
// deeper entries in private (scratch) memory, touched only by deep traversals.
// The LDS column is typed as LDS (address space 3) so that the compiler keeps
// LDS and private accesses apart: through a generic pointer it merges the two
// into one flat load, which waits on both memory counters.
typedef __attribute__((address_space(3))) int32_t lds_i32;
// Read by scalar loads where the address is the same in every lane.
typedef const __attribute__((address_space(4))) float const_f32;
typedef const __attribute__((address_space(4))) int32_t const_i32;

template <int LDS_DEPTH, int SIZE = kStackSize>
struct TraversalStack {
    static constexpr int kDeep = SIZE - LDS_DEPTH > 0 ? SIZE - LDS_DEPTH : 1;
    lds_i32* col;
    int32_t deep[kDeep];
    HX_DEV void put(int e, int32_t v) {
        if (e < LDS_DEPTH) col[e * kTraceBlock] = v;
        else deep[e - LDS_DEPTH] = v;
    }
    HX_DEV int32_t get(int e) const {
        if (e < LDS_DEPTH) return col[e * kTraceBlock];
        return deep[e - LDS_DEPTH];
    }
};

// Lanes that share a ray (SHARE).  When a wave's rays are all handed out, its
// idle lanes take stack entries of its busy lanes and traverse them for the same
// ray; the ray's best hit lives in the owner lane's slot.  (t, id) packs into
// one word whose order is "smaller t, then smaller id", the tie rule, so an LDS
// atomic minimum merges hits, and every lane adopts the best one once a round.
// The closest hit does not depend on which lane tests what.
// A ray is a serial chain of ~0.4 us a visit, hundreds of visits for the longest
// ones, so small ray sets and the end of every launch last as long as their
// longest rays: 4,096 rays 40 -> 26 us, 16,384 147 -> 49 us, 65,536 340 -> 182 us,
// 262,144 268 -> 225 us, 1,048,576 399 -> 365 us, 4.2M camera rays 1216 -> 1039 us.
// What is taken: while few lanes are busy the lowest entry, the largest subtree,
// which spreads the work fastest; else the top one, the next the lane would
// visit, since far subtrees are mostly culled once the near ones are done (always
// the lowest: 262,144 rays 332 us; always the top: 16,384 rays 77 us).
struct ShareSlot {
    uint64_t key;
    float2 uv;
};
// Orders this wave's LDS accesses (no instruction: the wave runs in lockstep).
HX_DEV void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }
constexpr int kShareLow = 16;     // busy lanes up to which the lowest entry is taken
constexpr int kShareVisits = 8;   // node visits between two rounds of sharing
HX_DEV uint64_t share_key(float t, int32_t id) {
    const uint32_t b = __float_as_uint(t);
    return (uint64_t)(b ^ (b >> 31 ? 0xFFFFFFFFu : 0x80000000u)) << 32 | (uint32_t)id;
}
HX_DEV void share_adopt(uint64_t key, float& t, int32_t& id, bool always = false) {
    if (!always && key >= share_key(t, id == -1 ? 0 : id)) return;
    const uint32_t b = (uint32_t)(key >> 32);
    t = __uint_as_float(b ^ (b >> 31 ? 0x80000000u : 0xFFFFFFFFu));
    id = (int32_t)(uint32_t)key;
}

// POSTPONE: leaves a lane may hold back while its wave still traverses (1, as
// HipTracerBinKernels.cu:169-177; 2 is the reference's commented variant,
// :171-173, 255; up to 4 here).  Held leaves wait in leafAddr (newest) ..
// leafAddr4; a lane whose slots are full stops until its wave has a leaf in
// every lane, or until at most half of the wave's live lanes still look for one
// (the lanes that wait cost more than the leaf phases saved: 16.7M diffuse rays
// 6.62 -> 6.26 ms, 2M any-hit rays 1.79 -> 1.52 ms).  The closest hit does not
// depend on the order leaves are tested; any-hit rays test theirs oldest first,
// which is traversal order, so that the hit they report is the same however
// many are held.
//
// A node is read by vector loads, which cost the CU's texture address and data
// units four 16-byte-per-lane instructions however many lanes share it.  With
// rays from one point (ALIKE) a node that all active lanes of the wave visit is
// read by scalar loads instead (constant address space: the trace never writes
// the nodes).  For other rays the check costs more than the reads it saves (16,384
// rays 10 %).
template <bool STATS, bool ORDERED, int LDS_DEPTH, int POSTPONE, int AHEAD, bool SHARE, bool ALIKE>
HX_TRACE_KERNEL __attribute__((amdgpu_waves_per_eu(LDS_DEPTH <= 16 ? 8 : 1))) void k_trace(TraceArgs a) {
    __shared__ int32_t s_stack[LDS_DEPTH > 0 ? LDS_DEPTH * kTraceBlock : 1];
    __shared__ ShareSlot s_share[SHARE ? kTraceBlock : 1];
    TraversalStack<LDS_DEPTH> stack;
    stack.col = (lds_i32*)(s_stack + threadIdx.x);
    int sp = 0;
    float ox = 0.f, oy = 0.f, oz = 0.f, tmin = 0.f, dx = 0.f, dy = 0.f, dz = 0.f;
    float idx = 0.f, idy = 0.f, idz = 0.f, oodx = 0.f, oody = 0.f, oodz = 0.f;
    float hitT = 0.f, hitU = 0.f, hitV = 0.f;
    int32_t nodeAddr = kSentinel, leafAddr = 0, leafAddr2 = 0, leafAddr3 = 0, leafAddr4 = 0, hitIndex = -1,
            hitId = -1;
    int32_t rayidx = -1;
    int32_t nNodes = 0, nTris = 0;
    // Batched trace: this lane's mesh (node base, first triangle position).
    int32_t nodeBase = 0, triBase = 0;
    const int lane = lane_id();
    if (!SHARE && lane >= a.lanes) return;
    const bool alike = ALIKE && __builtin_amdgcn_readfirstlane(a.control[kControlAlike]) != 0;
    RayPool pool;
    pool.start(a, alike);
    // SHARE, once the rays are handed out: lane whose ray this lane works on,
    // its slot, and this lane's lowest stack entry that may be given away.
    ShareSlot* const wave_slots = s_share + (SHARE ? threadIdx.x - lane : 0);
    bool sharing = false;
    int share = lane | 1 << 8;   // owner lane, lowest entry << 8

    while (true) {
        // Fetch new rays for the terminated lanes of this wave.
        const bool terminated = nodeAddr == kSentinel && (!SHARE || lane < a.lanes);
        if (!sharing) {
            const uint64_t tmask = ballot64(terminated);
            const int slot = pool.take(terminated, tmask, __popcll(tmask), a.control);
            if (terminated && (!SHARE || slot < (int)a.n_rays)) {
                if (!SHARE && slot >= (int)a.n_rays) break;
                rayidx = ORDERED ? a.order[slot] : slot;
                const int m = a.ray_mesh ? a.ray_mesh[rayidx] : 0;
                if (a.ray_mesh && (unsigned)m >= (unsigned)a.n_meshes) {  // no such mesh: a miss
                    reinterpret_cast<int2*>(a.results)[2 * (int64_t)rayidx] =
                        make_int2(-1, __float_as_int(a.rays[2 * (int64_t)rayidx + 1].w));
                    if (STATS) a.stats[rayidx] = make_int2(0, 0);
                    rayidx = -1;
                } else {
                    if (a.ray_mesh) {
                        nodeBase = a.mesh_tab[m].x;
                        triBase = a.mesh_off[m];
                    }
                    const float4 o = a.rays[2 * (int64_t)rayidx + 0];
                    const float4 d = a.rays[2 * (int64_t)rayidx + 1];
                    ox = o.x; oy = o.y; oz = o.z; tmin = o.w;
                    dx = d.x; dy = d.y; dz = d.z; hitT = d.w;
                    const float ooeps = 8.2718061255302767e-25f;  // exp2f(-80)
                    idx = 1.0f / (fabsf(dx) > ooeps ? dx : copysignf(ooeps, dx));
                    idy = 1.0f / (fabsf(dy) > ooeps ? dy : copysignf(ooeps, dy));
                    idz = 1.0f / (fabsf(dz) > ooeps ? dz : copysignf(ooeps, dz));
                    oodx = ox * idx;
                    oody = oy * idy;
                    oodz = oz * idz;
                    stack.put(0, kSentinel);
                    sp = 0;
                    leafAddr = 0;
                    leafAddr2 = 0;
                    leafAddr3 = 0;
                    leafAddr4 = 0;
                    nodeAddr = 0;
                    hitIndex = -1;
                    hitId = -1;
                    if (STATS) { nNodes = 0; nTris = 0; }
                }
            }
        }
        int visits = 0x7fffffff;
        if (SHARE && (sharing || (pool.next >= pool.end && pool.base >= pool.n))) {
            if (!sharing) {
                sharing = true;
                wave_slots[lane].key = share_key(hitT, hitIndex == -1 ? 0 : hitId);
                wave_slots[lane].uv = make_float2(hitU, hitV);
                hitIndex = -1;
            }
            ShareSlot* const mine = wave_slots + (share & 0xFF);
            wave_fence();
            if (hitIndex != -1) {   // a hit since the last round
                const uint64_t key = share_key(hitT, hitId);
                // A ray that may hit at t <= 0 is not shared: -0 and 0 tie, but
                // not as keys.
                if (tmin >= 0.0f) __hip_atomic_fetch_min(&mine->key, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                else mine->key = key;
                wave_fence();
                if (mine->key == key) mine->uv = make_float2(hitU, hitV);
                hitIndex = -1;
            }
            wave_fence();
            const uint64_t busy = ballot64(nodeAddr != kSentinel);
            if (!busy) break;
            // The best hit of the ray so far, whoever found it.
            if (nodeAddr != kSentinel) share_adopt(mine->key, hitT, hitId);
            // The k-th idle lane takes the lowest stack entry of the k-th lane that has one.
            const bool low = __popcll(busy) <= kShareLow;
            const bool gives = nodeAddr != kSentinel && (share >> 8) <= sp && (low ? share >> 8 : sp) < LDS_DEPTH && tmin >= 0.0f;
            const uint64_t gm = ballot64(gives);
            const uint64_t im = ~busy;
            const int pairs = min(__popcll(gm), __popcll(im));
            if (pairs > 0 && __popcll(busy) <= a.share_busy) {
                const int grank = count_below(gm), irank = count_below(im);
                // Lane k learns the k-th giving lane.
                const int kth = __builtin_amdgcn_ds_permute((gives ? grank : 63) << 2, lane);
                const bool takes = nodeAddr == kSentinel && irank < pairs;
                const int from = __shfl(kth, takes ? irank : 0, kWave);
                const int e = __shfl(low ? share >> 8 : sp, from, kWave);
                lds_i32* const src = stack.col - lane + from + e * kTraceBlock;
                int32_t got = 0;
                if (takes) {
                    got = *src;
                    if (low) *src = kSentinel;
                }
                if (gives && grank < pairs) {
                    if (low) share += 1 << 8;
                    else --sp;
                }
                auto copy = [&](auto& v) {
                    const auto x = __shfl(v, from, kWave);
                    if (takes) v = x;
                };
                copy(ox); copy(oy); copy(oz); copy(tmin);
                copy(dx); copy(dy); copy(dz);
                copy(idx); copy(idy); copy(idz);
                copy(oodx); copy(oody); copy(oodz);
                copy(hitT); copy(hitId); copy(share);
                if (takes) {
                    nodeAddr = got;
                    leafAddr = leafAddr2 = leafAddr3 = leafAddr4 = 0;
                    stack.put(0, kSentinel);
                    sp = 0;
                    share = (share & 0xFF) | 1 << 8;
                }
            }
            wave_fence();
            visits = kShareVisits;
        }

        while (nodeAddr != kSentinel) {
            if (SHARE && nodeAddr < 0) {   // a leaf that was handed over: nothing else is on the stack
                leafAddr = nodeAddr;
                nodeAddr = kSentinel;
            }
            const int half = __popcll(ballot64(true)) >> 1;
            int left = visits;
            while ((uint32_t)nodeAddr < (uint32_t)kSentinel) {
                if (STATS) ++nNodes;
                float c0min, c0max, c1min, c1max;
                int2 cn;
                // Written out in both branches below, so that a node of the whole
                // wave is tested straight from the scalar registers.
                auto box_test = [&](float4 n0xy, float4 n1xy, float4 nz) {
                    const float c0lox = fmaf(n0xy.x, idx, -oodx);
                    const float c0hix = fmaf(n0xy.y, idx, -oodx);
                    const float c0loy = fmaf(n0xy.z, idy, -oody);
                    const float c0hiy = fmaf(n0xy.w, idy, -oody);
                    const float c0loz = fmaf(nz.x, idz, -oodz);
                    const float c0hiz = fmaf(nz.y, idz, -oodz);
                    const float c1loz = fmaf(nz.z, idz, -oodz);
                    const float c1hiz = fmaf(nz.w, idz, -oodz);
                    c0min = span_begin(c0lox, c0hix, c0loy, c0hiy, c0loz, c0hiz, tmin);
                    c0max = span_end(c0lox, c0hix, c0loy, c0hiy, c0loz, c0hiz, hitT);
                    const float c1lox = fmaf(n1xy.x, idx, -oodx);
                    const float c1hix = fmaf(n1xy.y, idx, -oodx);
                    const float c1loy = fmaf(n1xy.z, idy, -oody);
                    const float c1hiy = fmaf(n1xy.w, idy, -oody);
                    c1min = span_begin(c1lox, c1hix, c1loy, c1hiy, c1loz, c1hiz, tmin);
                    c1max = span_end(c1lox, c1hix, c1loy, c1hiy, c1loz, c1hiz, hitT);
                };
                const uint32_t na = (uint32_t)(nodeBase + nodeAddr);
                const uint32_t n0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)na);
                if (alike && __all(na == n0)) {
                    const_f32* f = (const_f32*)(a.nodes + 4 * (int64_t)n0);
                    const_i32* w = (const_i32*)(a.nodes + 4 * (int64_t)n0);
                    box_test(make_float4(f[0], f[1], f[2], f[3]), make_float4(f[4], f[5], f[6], f[7]),
                             make_float4(f[8], f[9], f[10], f[11]));
                    cn = make_int2(w[12], w[13]);
                } else {
                    const float4* np = reinterpret_cast<const float4*>(a.nodes + 4 * (int64_t)na);
                    const float4 n0xy = np[0];
                    const float4 n1xy = np[1];
                    const float4 nz = np[2];
                    const int4 links = a.nodes[4 * (int64_t)na + 3];
                    // The child links share the node's cache line: keep their
                    // load with the box loads instead of after the box test.
                    asm volatile("" ::"v"(links.x), "v"(links.y));
                    cn = make_int2(links.x, links.y);
                    box_test(n0xy, n1xy, nz);
                }
                const bool swp = c1min < c0min;
                const bool t0 = c0max >= c0min;
                const bool t1 = c1max >= c1min;
                int32_t cy = cn.y;
                if (!t0 && !t1) {
                    nodeAddr = stack.get(sp--);
                } else {
                    nodeAddr = t0 ? cn.x : cy;
                    if (t0 && t1) {
                        if (swp) {
                            const int32_t tmp = nodeAddr;
                            nodeAddr = cy;
                            cy = tmp;
                        }
                        if (sp + 1 >= kStackSize) {
                            atomicAdd(a.control + 1, 1);
                            nodeAddr = kSentinel;
                            leafAddr = leafAddr2 = leafAddr3 = leafAddr4 = 0;
                            break;
                        }
                        stack.put(++sp, cy);
                    }
                }
                const int32_t lastSlot = POSTPONE == 1 ? leafAddr : POSTPONE == 2 ? leafAddr2
                                         : POSTPONE == 3 ? leafAddr3 : leafAddr4;
                if (nodeAddr < 0 && lastSlot >= 0) {
                    if (a.any_hit) {
                        const bool h1 = leafAddr < 0, h2 = leafAddr2 < 0, h3 = leafAddr3 < 0;
                        if (POSTPONE >= 4) leafAddr4 = h3 ? nodeAddr : 0;
                        if (POSTPONE >= 3) leafAddr3 = h2 && !h3 ? nodeAddr : leafAddr3;
                        if (POSTPONE >= 2) leafAddr2 = h1 && !h2 ? nodeAddr : leafAddr2;
                        leafAddr = h1 ? leafAddr : nodeAddr;
                    } else {
                        if (POSTPONE >= 4) leafAddr4 = leafAddr3;
                        if (POSTPONE >= 3) leafAddr3 = leafAddr2;
                        if (POSTPONE >= 2) leafAddr2 = leafAddr;
                        leafAddr = nodeAddr;
                    }
                    nodeAddr = stack.get(sp--);
                }
                if (!__any(leafAddr >= 0) || __popcll(ballot64(true)) <= half) break;
                if (SHARE && --left == 0) break;
            }

            while (leafAddr < 0) {
                const int4 lb = a.nodes[4 * (int64_t)(uint32_t)(nodeBase + ~leafAddr) + 3];
                // The next triangle's first Woop row (AHEAD = 1), or its first
                // two (AHEAD = 2), are read while this one is tested: leaves of
                // long thin triangles test hundreds per ray, and most of those
                // tests pass the plane test and need the second row.
                const float4* wrow = a.woop + 3 * (int64_t)(triBase + lb.x);
                float4 vnext = lb.x < lb.y ? wrow[0] : make_float4(0.f, 0.f, 0.f, 0.f);
                float4 vnext1 = AHEAD >= 2 && lb.x < lb.y ? wrow[1] : make_float4(0.f, 0.f, 0.f, 0.f);
                for (int tri = lb.x; tri < lb.y; ++tri, wrow += 3) {
                    if (STATS) ++nTris;
                    const float4 v00 = vnext;
                    const float4 v11n = vnext1;
                    if (tri + 1 < lb.y) {
                        vnext = wrow[3];
                        if (AHEAD >= 2) vnext1 = wrow[4];
                    }
                    const float Oz = fmaf(-oz, v00.z, fmaf(-oy, v00.y, fmaf(-ox, v00.x, v00.w)));
                    const float den = fmaf(dz, v00.z, fmaf(dy, v00.y, dx * v00.x));
                    const float t = Oz * (1.0f / den);
                    if (t > tmin && t <= hitT) {
                        const float4 v11 = AHEAD >= 2 ? v11n : wrow[1];
                        const float Ox = fmaf(oz, v11.z, fmaf(oy, v11.y, fmaf(ox, v11.x, v11.w)));
                        const float Dx = fmaf(dz, v11.z, fmaf(dy, v11.y, dx * v11.x));
                        const float u = fmaf(t, Dx, Ox);
                        if (u >= 0.0f) {
                            const float4 v22 = wrow[2];
                            const float Oy = fmaf(oz, v22.z, fmaf(oy, v22.y, fmaf(ox, v22.x, v22.w)));
                            const float Dy = fmaf(dz, v22.z, fmaf(dy, v22.y, dx * v22.x));
                            const float v = fmaf(t, Dy, Oy);
                            if (v >= 0.0f && u + v <= 1.0f) {
                                const int32_t id = a.tri_idx[triBase + tri];
                                // Closest hit; equal t resolves to the smaller triangle id.
                                if (t < hitT || id < hitId) {
                                    hitT = t;
                                    hitIndex = tri;
                                    hitId = id;
                                    hitU = u;
                                    hitV = v;
                                    if (a.any_hit) {
                                        nodeAddr = kSentinel;
                                        leafAddr2 = leafAddr3 = leafAddr4 = 0;
                                        break;
                                    }
                                }
                            }
                        }
                    }
                }
                if (POSTPONE >= 2 && leafAddr2 < 0) {  // the other held leaves next
                    leafAddr = leafAddr2;
                    leafAddr2 = POSTPONE >= 3 ? leafAddr3 : 0;
                    leafAddr3 = POSTPONE >= 4 ? leafAddr4 : 0;
                    leafAddr4 = 0;
                } else {
                    leafAddr = nodeAddr;
                    if (nodeAddr < 0) nodeAddr = stack.get(sp--);
                }
            }

            if (__popcll(ballot64(true)) < a.fetch_threshold || (SHARE && sharing)) break;
        }

        if (nodeAddr == kSentinel && rayidx >= 0 && !(SHARE && sharing)) {
            if (hitIndex == -1)
                reinterpret_cast<int2*>(a.results)[2 * (int64_t)rayidx] = make_int2(-1, __float_as_int(hitT));
            else
                a.results[rayidx] =
                    make_int4(hitId, __float_as_int(hitT), __float_as_int(hitU), __float_as_int(hitV));
            if (STATS) a.stats[rayidx] = make_int2(nNodes, nTris);
            rayidx = -1;
        }
    }
    if (SHARE && rayidx >= 0) {
        const ShareSlot r = wave_slots[lane];
        const float tmax = a.rays[2 * (int64_t)rayidx + 1].w;
        if (r.key == share_key(tmax, 0)) {
            reinterpret_cast<int2*>(a.results)[2 * (int64_t)rayidx] = make_int2(-1, __float_as_int(tmax));
        } else {
            float t = 0.0f;
            int32_t id = 0;
            share_adopt(r.key, t, id, true);
            a.results[rayidx] = make_int4(id, __float_as_int(t), __float_as_int(r.uv.x), __float_as_int(r.uv.y));
        }
    }
}

// ---------------------------------------------------------------------------
// Quad / Oct traversal (HipTracerQuadKernels.cu, HipTracerOctKernels.cu; node
// words of HipBVHNode.h:13-114).  One ray per lane, as the Bin kernel: a node
// visit tests its N child boxes (child c: float4 c = min/max x, min/max y;
// float4 N + c = min/max z, link), sorts the hits by entry distance with a
// compare-exchange network in registers (ties by link), continues into the
// nearest and pushes the others farthest first.  The reference gives each
// ray N lanes; on 64-lane waves that leaves 64/N rays per wave to hide each
// node fetch, so here every lane keeps its own ray and the waves stay full.
// Leaves (link ~index) hold [begin, end) at words 4N+2, 4N+3; the triangle
// test, closest-hit tie rule, postponed leaf and wave refill are the Bin
// kernel's.
// ---------------------------------------------------------------------------

template <int N>
struct WideNet;
template <>
struct WideNet<4> {
    static constexpr int kPairs = 5;
    HX_DEV static int2 pair(int i) {
        constexpr int a[5] = {0, 2, 0, 1, 1}, b[5] = {1, 3, 2, 3, 2};
        return make_int2(a[i], b[i]);
    }
};
template <>
struct WideNet<8> {
    // Batcher's odd-even merge sort for 8 inputs.
    static constexpr int kPairs = 19;
    HX_DEV static int2 pair(int i) {
        constexpr int a[19] = {0, 2, 4, 6, 0, 1, 4, 5, 1, 5, 0, 1, 2, 3, 2, 3, 1, 3, 5};
        constexpr int b[19] = {1, 3, 5, 7, 2, 3, 6, 7, 2, 6, 4, 5, 6, 7, 4, 5, 2, 4, 6};
        return make_int2(a[i], b[i]);
    }
};

template <int N>
struct WideStackSize {
    static constexpr int kSize = N == 4 ? 96 : 160;
};

template <int N, bool STATS, bool ORDERED, int LDS_DEPTH, bool ALIKE>
HX_TRACE_KERNEL void k_trace_wide(TraceArgs a) {
    constexpr int kSize = WideStackSize<N>::kSize;
    __shared__ int32_t s_stack[LDS_DEPTH > 0 ? LDS_DEPTH * kTraceBlock : 1];
    TraversalStack<LDS_DEPTH, kSize> stack;
    stack.col = (lds_i32*)(s_stack + threadIdx.x);
    int sp = 0;
    float ox = 0.f, oy = 0.f, oz = 0.f, tmin = 0.f, dx = 0.f, dy = 0.f, dz = 0.f;
    float idx = 0.f, idy = 0.f, idz = 0.f, oodx = 0.f, oody = 0.f, oodz = 0.f;
    float hitT = 0.f, hitU = 0.f, hitV = 0.f;
    int32_t nodeAddr = kSentinel, leafAddr = 0, hitIndex = -1, hitId = -1;
    int64_t rayidx = 0;
    int32_t nNodes = 0, nTris = 0;
    const float4* nodes4 = reinterpret_cast<const float4*>(a.nodes);
    if (lane_id() >= a.lanes) return;
    const bool alike = ALIKE && __builtin_amdgcn_readfirstlane(a.control[kControlAlike]) != 0;
    RayPool pool;
    pool.start(a, alike);

    while (true) {
        const bool terminated = nodeAddr == kSentinel;
        const uint64_t tmask = ballot64(terminated);
        const int slot = pool.take(terminated, tmask, __popcll(tmask), a.control);
        if (terminated) {
            rayidx = slot;
            if (rayidx >= a.n_rays) break;
            if (ORDERED) rayidx = a.order[rayidx];
            const float4 o = a.rays[2 * rayidx + 0];
            const float4 d = a.rays[2 * rayidx + 1];
            ox = o.x; oy = o.y; oz = o.z; tmin = o.w;
            dx = d.x; dy = d.y; dz = d.z; hitT = d.w;
            const float ooeps = 8.2718061255302767e-25f;  // exp2f(-80)
            idx = 1.0f / (fabsf(dx) > ooeps ? dx : copysignf(ooeps, dx));
            idy = 1.0f / (fabsf(dy) > ooeps ? dy : copysignf(ooeps, dy));
            idz = 1.0f / (fabsf(dz) > ooeps ? dz : copysignf(ooeps, dz));
            oodx = ox * idx;
            oody = oy * idy;
            oodz = oz * idz;
            stack.put(0, kSentinel);
            sp = 0;
            leafAddr = 0;
            nodeAddr = 0;
            hitIndex = -1;
            hitId = -1;
            if (STATS) { nNodes = 0; nTris = 0; }
        }
        while (nodeAddr != kSentinel) {
            const int half = __popcll(ballot64(true)) >> 1;
            while ((uint32_t)nodeAddr < (uint32_t)kSentinel) {
                if (STATS) ++nNodes;
                float dist[N];
                int32_t link[N];
                // Child c's test; written out in both node-read branches, as in k_trace.
                auto child_test = [&](int c, float4 xy, float4 zl) {
                    const float lox = fmaf(xy.x, idx, -oodx);
                    const float hix = fmaf(xy.y, idx, -oodx);
                    const float loy = fmaf(xy.z, idy, -oody);
                    const float hiy = fmaf(xy.w, idy, -oody);
                    const float loz = fmaf(zl.x, idz, -oodz);
                    const float hiz = fmaf(zl.y, idz, -oodz);
                    const float cmin = span_begin(lox, hix, loy, hiy, loz, hiz, tmin);
                    const float cmax = span_end(lox, hix, loy, hiy, loz, hiz, hitT);
                    const bool hit = cmax >= cmin;
                    dist[c] = hit ? cmin : __int_as_float(0x7f800000);
                    link[c] = hit ? __float_as_int(zl.z) : kSentinel;
                };
                const int32_t n0 = __builtin_amdgcn_readfirstlane(nodeAddr);
                if (alike && __all(nodeAddr == n0)) {
                    const_f32* f = (const_f32*)(nodes4 + (int64_t)n0 * 2 * N);
#pragma unroll
                    for (int c = 0; c < N; ++c)
                        child_test(c, make_float4(f[4 * c], f[4 * c + 1], f[4 * c + 2], f[4 * c + 3]),
                                   make_float4(f[4 * (N + c)], f[4 * (N + c) + 1], f[4 * (N + c) + 2],
                                               f[4 * (N + c) + 3]));
                } else {
                    const float4* np = nodes4 + (int64_t)nodeAddr * 2 * N;
                    float4 xys[N], zls[N];
#pragma unroll
                    for (int c = 0; c < N; ++c) {
                        xys[c] = np[c];
                        zls[c] = np[N + c];
                    }
#pragma unroll
                    for (int c = 0; c < N; ++c) child_test(c, xys[c], zls[c]);
                }
#pragma unroll
                for (int q = 0; q < WideNet<N>::kPairs; ++q) {
                    const int2 pr = WideNet<N>::pair(q);
                    const float da = dist[pr.x], db = dist[pr.y];
                    const int32_t la = link[pr.x], lb = link[pr.y];
                    const bool sw = db < da || (db == da && lb < la);
                    dist[pr.x] = sw ? db : da;
                    dist[pr.y] = sw ? da : db;
                    link[pr.x] = sw ? lb : la;
                    link[pr.y] = sw ? la : lb;
                }
                int cnt = 0;
#pragma unroll
                for (int c = 0; c < N; ++c) cnt += link[c] != kSentinel ? 1 : 0;
                if (cnt == 0) {
                    nodeAddr = stack.get(sp--);
                } else {
                    if (sp + cnt >= kSize) {
                        atomicAdd(a.control + 1, 1);
                        nodeAddr = kSentinel;
                        leafAddr = 0;
                        break;
                    }
#pragma unroll
                    for (int c = N - 1; c >= 1; --c)
                        if (c < cnt) stack.put(++sp, link[c]);
                    nodeAddr = link[0];
                }
                if (nodeAddr < 0 && leafAddr >= 0) {
                    leafAddr = nodeAddr;
                    nodeAddr = stack.get(sp--);
                }
                if (!__any(leafAddr >= 0) || __popcll(ballot64(true)) <= half) break;
            }

            while (leafAddr < 0) {
                const float4 lb = nodes4[(int64_t)(~leafAddr) * 2 * N + N];
                const int end = __float_as_int(lb.w);
                for (int tri = __float_as_int(lb.z); tri < end; ++tri) {
                    if (STATS) ++nTris;
                    const float4 v00 = a.woop[3 * (int64_t)tri + 0];
                    const float Oz = fmaf(-oz, v00.z, fmaf(-oy, v00.y, fmaf(-ox, v00.x, v00.w)));
                    const float den = fmaf(dz, v00.z, fmaf(dy, v00.y, dx * v00.x));
                    const float t = Oz * (1.0f / den);
                    if (t > tmin && t <= hitT) {
                        const float4 v11 = a.woop[3 * (int64_t)tri + 1];
                        const float Ox = fmaf(oz, v11.z, fmaf(oy, v11.y, fmaf(ox, v11.x, v11.w)));
                        const float Dx = fmaf(dz, v11.z, fmaf(dy, v11.y, dx * v11.x));
                        const float u = fmaf(t, Dx, Ox);
                        if (u >= 0.0f) {
                            const float4 v22 = a.woop[3 * (int64_t)tri + 2];
                            const float Oy = fmaf(oz, v22.z, fmaf(oy, v22.y, fmaf(ox, v22.x, v22.w)));
                            const float Dy = fmaf(dz, v22.z, fmaf(dy, v22.y, dx * v22.x));
                            const float v = fmaf(t, Dy, Oy);
                            if (v >= 0.0f && u + v <= 1.0f) {
                                const int32_t id = a.tri_idx[tri];
                                // Closest hit; equal t resolves to the smaller triangle id.
                                if (t < hitT || id < hitId) {
                                    hitT = t;
                                    hitIndex = tri;
                                    hitId = id;
                                    hitU = u;
                                    hitV = v;
                                    if (a.any_hit) {
                                        nodeAddr = kSentinel;
                                        break;
                                    }
                                }
                            }
                        }
                    }
                }
                leafAddr = nodeAddr;
                if (nodeAddr < 0) nodeAddr = stack.get(sp--);
            }

            if (__popcll(ballot64(true)) < a.fetch_threshold) break;
        }

        if (nodeAddr == kSentinel) {
            if (hitIndex == -1)
                reinterpret_cast<int2*>(a.results)[2 * rayidx] = make_int2(-1, __float_as_int(hitT));
            else
                a.results[rayidx] =
                    make_int4(hitId, __float_as_int(hitT), __float_as_int(hitU), __float_as_int(hitV));
            if (STATS) a.stats[rayidx] = make_int2(nNodes, nTris);
        }
    }
}

// ---------------------------------------------------------------------------
// Ray Morton keys for the [0,1]^3 ray box (RayBuffer.cpp:63-66).
// ---------------------------------------------------------------------------

HX_DEV float fmin_n(float a, float b) { return (a != a) ? b : (b != b) ? a : ((b < a) ? b : a); }
HX_DEV float fmax_n(float a, float b) { return (a != a) ? b : (b != b) ? a : ((b > a) ? b : a); }

__global__ void k_ray_keys_aila(const float4* __restrict__ rays, int64_t n, int bits, uint64_t* __restrict__ keys) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 o = rays[2 * i], d = rays[2 * i + 1];
    const float ax = (o.x - 0.0f) / (1.0f - 0.0f), ay = (o.y - 0.0f) / (1.0f - 0.0f), az = (o.z - 0.0f) / (1.0f - 0.0f);
    float ls = 0.0f;
    ls += d.x * d.x;
    ls += d.y * d.y;
    ls += d.z * d.z;
    const float len = sqrtf(ls);
    const float rl = (len != 0.0f) ? 1.0f / len : 0.0f;
    const float bx = (d.x * rl + 1.0f) * 0.5f, by = (d.y * rl + 1.0f) * 0.5f, bz = (d.z * rl + 1.0f) * 0.5f;
    const int iax = f2i_sat(ax * 8191.0f), iay = f2i_sat(ay * 8191.0f), iaz = f2i_sat(az * 8191.0f);
    const int ibx = f2i_sat(bx * 8191.0f), iby = f2i_sat(by * 8191.0f), ibz = f2i_sat(bz * 8191.0f);
    uint64_t code = 0;
    code |= (uint64_t)((iax >> 12) & 1) << 63;
    code |= (uint64_t)((iay >> 12) & 1) << 62;
    code |= (uint64_t)((iaz >> 12) & 1) << 61;
    code |= (uint64_t)((iax >> 11) & 1) << 60;
    code |= (uint64_t)((iay >> 11) & 1) << 59;
    code |= (uint64_t)((iaz >> 11) & 1) << 58;
    code |= (uint64_t)((iax >> 10) & 1) << 57;
    code |= (uint64_t)((iay >> 10) & 1) << 56;
    code |= (uint64_t)((iaz >> 10) & 1) << 55;
#pragma unroll
    for (int k = 9; k >= 1; --k) {
        code |= (uint64_t)((iax >> k) & 1) << (6 * k + 0);
        code |= (uint64_t)((iay >> k) & 1) << (6 * k - 1);
        code |= (uint64_t)((iaz >> k) & 1) << (6 * k - 2);
    }
#pragma unroll
    for (int k = 12; k >= 4; --k) {
        code |= (uint64_t)((ibx >> k) & 1) << (6 * k - 21);
        code |= (uint64_t)((iby >> k) & 1) << (6 * k - 22);
        code |= (uint64_t)((ibz >> k) & 1) << (6 * k - 23);
    }
    keys[i] = code >> (64 - bits);
}

__global__ void k_ray_keys_twopoint(const float4* __restrict__ rays, int64_t n, int bits, float ray_length,
                                    uint64_t* __restrict__ keys) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 ro = rays[2 * i], rd = rays[2 * i + 1];
    const float o[3] = {ro.x, ro.y, ro.z}, d[3] = {rd.x, rd.y, rd.z};
    float tmn[3], tmx[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (d[k] >= 0.0f) {
            tmn[k] = (0.0f - o[k]) / d[k];
            tmx[k] = (1.0f - o[k]) / d[k];
        } else {
            tmn[k] = (1.0f - o[k]) / d[k];
            tmx[k] = (0.0f - o[k]) / d[k];
        }
    }
    const float t0 = fmax_n(tmn[2], fmax_n(tmn[0], tmn[1]));
    const float t1 = fmin_n(tmx[2], fmin_n(tmx[0], tmx[1]));
    const float boxT = (t0 > t1) ? -1.0f : (1.0f - 1.0e-3f) * (t0 >= 0.0f ? t0 : t1);
    float len = ray_length;
    len = fmin_n(len, fmax_n(rd.w, 0.0f));
    len = fmin_n(len, boxT);
    int ia[3], ib[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float av = (o[k] - 0.0f) * (1.0f / (1.0f - 0.0f));
        const float bv = ((o[k] + len * d[k]) - 0.0f) * (1.0f / (1.0f - 0.0f));
        ia[k] = f2i_sat(av * 8191.0f);
        ib[k] = f2i_sat(bv * 8191.0f);
    }
    uint64_t code = 0;
#pragma unroll
    for (int k = 12; k >= 2; --k) {
        code |= (uint64_t)((ia[0] >> k) & 1) << (6 * k - 9);
        code |= (uint64_t)((ia[1] >> k) & 1) << (6 * k - 10);
        code |= (uint64_t)((ia[2] >> k) & 1) << (6 * k - 11);
    }
#pragma unroll
    for (int k = 12; k >= 3; --k) {
        code |= (uint64_t)((ib[0] >> k) & 1) << (6 * k - 12);
        code |= (uint64_t)((ib[1] >> k) & 1) << (6 * k - 13);
        code |= (uint64_t)((ib[2] >> k) & 1) << (6 * k - 14);
    }
    code |= (uint64_t)(ib[0] & 1);
    keys[i] = code >> (64 - bits);
}

__global__ void k_zero_control(int32_t* control) {
    if (threadIdx.x < 2) control[threadIdx.x] = 0;
}

// k_zero_control of a launch that may hold rays from one point: kAlikeWindows
// windows of 64 neighbouring rays, spread evenly over the set as it is traced.
// control[kControlAlike] is set if in more than half of them every ray is live (a
// dead one, with an empty interval, ends at once whatever its origin: the secondary
// rays of misses) and starts at the same point.
constexpr int kAlikeBlock = 1024, kAlikeWindows = 16;
__global__ __launch_bounds__(kAlikeBlock) void k_zero_control_alike(TraceArgs a) {
    __shared__ int s_alike[kAlikeBlock / kWave];
    const int w = threadIdx.x / kWave;
    static_assert(kAlikeWindows == kAlikeBlock / kWave, "one window a wave");
    const int64_t slot = (a.n_rays - kWave) * w / (kAlikeWindows - 1) + lane_id();
    const int64_t ray = a.order ? a.order[slot] : slot;
    const float4 o = a.rays[2 * ray], d = a.rays[2 * ray + 1];
    auto first = [](float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); };
    int count = __all(o.x == first(o.x) && o.y == first(o.y) && o.z == first(o.z) && d.w > o.w) ? 1 : 0;
    if (lane_id() == 0) s_alike[w] = count;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 1; k < kAlikeBlock / kWave; ++k) count += s_alike[k];
    a.control[0] = a.control[1] = 0;
    a.control[kControlAlike] = 2 * count > kAlikeWindows ? 1 : 0;
}

// Large sets are looked over for rays from one point (k_zero_control_alike; RayPool
// and k_trace say what they get): sorted sets from 2 rays a lane slot on (1.05M;
// any-hit rays, which seldom share an origin, from 4: the look costs 2.0M of them
// 0.8 %), from 4 in the wide kernels (2.1M), from 12 in input order (6.3M).  Below, and where half of
// the rays miss at the root, the one ray counter would set the pace: unsorted
// 1,048,576 rays over 65,536 triangles 359 -> 369 us, a step with 4.2M camera rays
// over 1.3M triangles 1.75 -> 1.79 ms.  Primaries of the Gaussian mixture and ground
// grid, refill by refill with scalar reads against runs with vector reads: 16.7M
// sorted rays over 16.7M / 1M / 65k triangles 6.39 -> 4.82, 7.79 -> 6.46, 4.15 ->
// 3.49 ms (Quad, 16.7M and 65k: 6.79 -> 4.98, 4.51 -> 3.48; Oct: 9.14 -> 7.01, 5.30 ->
// 4.30), 4.2M sorted 2.04 -> 1.53, 2.38 -> 2.02, 1.27 -> 1.04 ms, 1.05M sorted 0.83 ->
// 0.68, 0.92 -> 0.80, 0.47 -> 0.42 ms, 16.7M in input order 6.24 -> 5.15, 7.78 -> 7.02,
// 4.14 -> 3.52 ms.  Of the 1.6 ms at 16.7M triangles the hand-out gives 0.7 ms, the
// scalar reads 0.9.  The diffuse rays of these scenes take what they took (16.7M: 9.83,
// 10.4, 3.75 ms).  The counts of a stats trace keep to one kernel.
bool alike_pays(const Context* c, const TraceArgs& a, bool wide) {
    return !a.stats && a.n_rays >= (int64_t)c->cu_count * 8 * kTraceBlock *
                                      (wide ? 4 : !a.order ? 12 : a.any_hit ? 4 : 2);
}

int zero_control(Context* c, const TraceArgs& a, bool wide) {
    if (alike_pays(c, a, wide))
        hipLaunchKernelGGL(k_zero_control_alike, dim3(1), dim3(kAlikeBlock), 0, c->stream, a);
    else
        hipLaunchKernelGGL(k_zero_control, dim3(1), dim3(64), 0, c->stream, a.control);
    return check_launch("zero_control");
}

// Rays per wave, workgroups and run lengths of a launch.  A wave costs the same
// whether 16 or 64 of its lanes carry rays, and lanes that diverge wait for each
// other, so a launch that cannot fill the chip with full waves spreads its rays
// over more of them: half as many rays per wave while that still leaves waves
// idle, down to 16 (65,536 rays over 1M triangles 500 -> 357 us, 16,384 over
// 64k 187 -> 157 us; 8 or 4 rays per wave were slower, 484 us, since the address
// units take 4 lanes a cycle and neighbouring rays share nodes), or 8 where the
// other lanes share the rays (16,384 rays 60 -> 49 us).  While every wave has
// such lanes from the start they join at once; later, when the chip is full,
// only once half a wave is idle (262,144 rays 259 -> 225 us).
unsigned trace_shape(Context* c, int occ, bool share, TraceArgs& a) {
    const int per_cu = c->tune.trace_blocks_per_cu > 0 ? std::min(c->tune.trace_blocks_per_cu, occ) : occ;
    const int64_t waves = (int64_t)c->cu_count * per_cu * (kTraceBlock / kWave);
    a.lanes = kWave;
    const int least = share ? 8 : 16;
    while (a.lanes > least && a.n_rays <= waves * (a.lanes / 2)) a.lanes /= 2;
    a.share_busy = a.n_rays <= waves * 16 ? kWave : kWave / 2;
    a.run_shift = 2;
    while (((int64_t)1 << (a.run_shift - 2)) < waves) ++a.run_shift;
    a.fetch_threshold = std::max(1, a.fetch_threshold * a.lanes / kWave);
    const int64_t per_block = (int64_t)a.lanes * (kTraceBlock / kWave);
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((int64_t)c->cu_count * per_cu,
                                                            (a.n_rays + per_block - 1) / per_block));
}

// Sharing pays where the longest rays show: up to 16 rays a lane slot.  Above
// (16.7M rays and more) the tail is too short a part of the launch (sorted
// primaries over a Gaussian mixture of 16.7M triangles 3.19 -> 3.23 ms).  Batched rays lose by it (1.37M: 1131 -> 1187 us or
// more): they are short and hit early.  An any-hit trace reports the first hit of
// one lane's traversal order, and the counts of a stats trace are per ray.
bool share_pays(const Context* c, const TraceArgs& a) {
    return !a.any_hit && !a.stats && !a.ray_mesh && a.n_rays <= (int64_t)c->cu_count * 8 * kTraceBlock * 16;
}

template <bool STATS, bool ORDERED, int LDS_DEPTH, int POSTPONE, int AHEAD, bool SHARE, bool ALIKE>
int launch_trace_kernel(Context* c, const TraceArgs& a) {
    // Occupancy limit of this instantiation, queried once per process.
    static int occ = 0;
    if (occ == 0) {
        int q = 0;
        HX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&q, k_trace<STATS, ORDERED, LDS_DEPTH, POSTPONE, AHEAD, SHARE, ALIKE>,
                                                             kTraceBlock, 0));
        occ = std::max(q, 1);
    }
    TraceArgs t = a;
    const unsigned blocks = trace_shape(c, occ, SHARE, t);
    hipLaunchKernelGGL((k_trace<STATS, ORDERED, LDS_DEPTH, POSTPONE, AHEAD, SHARE, ALIKE>), dim3(blocks), dim3(kTraceBlock), 0,
                       c->stream, t);
    return check_launch("trace");
}

template <bool STATS, bool ORDERED, int LDS_DEPTH, int POSTPONE, int AHEAD, bool SHARE>
int launch_trace_t(Context* c, const TraceArgs& a) {
    if (!STATS && alike_pays(c, a, false))
        return launch_trace_kernel<false, ORDERED, LDS_DEPTH, POSTPONE, AHEAD, SHARE, true>(c, a);
    return launch_trace_kernel<STATS, ORDERED, LDS_DEPTH, POSTPONE, AHEAD, SHARE, false>(c, a);
}

template <bool STATS, bool ORDERED, int POSTPONE, int AHEAD>
int launch_trace_depth(Context* c, const TraceArgs& a) {
    switch (c->tune.trace_lds_stack) {
        case 0: return launch_trace_t<STATS, ORDERED, 0, POSTPONE, AHEAD, false>(c, a);
        case 16:
            if (!STATS && share_pays(c, a))
                return launch_trace_t<false, ORDERED, 16, POSTPONE, AHEAD, true>(c, a);
            return launch_trace_t<STATS, ORDERED, 16, POSTPONE, AHEAD, false>(c, a);
        case 24: return launch_trace_t<STATS, ORDERED, 24, POSTPONE, AHEAD, false>(c, a);
        case 32: return launch_trace_t<STATS, ORDERED, 32, POSTPONE, AHEAD, false>(c, a);
        default: return launch_trace_t<STATS, ORDERED, 64, POSTPONE, AHEAD, false>(c, a);
    }
}

template <bool STATS, bool ORDERED, int POSTPONE>
int launch_trace_ahead(Context* c, const TraceArgs& a) {
    if (c->tune.trace_woop_ahead >= 2) return launch_trace_depth<STATS, ORDERED, POSTPONE, 2>(c, a);
    return launch_trace_depth<STATS, ORDERED, POSTPONE, 1>(c, a);
}

template <bool STATS, bool ORDERED>
int launch_trace_postpone(Context* c, const TraceArgs& a) {
    // Counts of an any-hit trace stay those of the reference's one postponed leaf.
    if (STATS && a.any_hit) return launch_trace_ahead<STATS, ORDERED, 1>(c, a);
    switch (c->tune.trace_postpone) {
        case 2: return launch_trace_ahead<STATS, ORDERED, 2>(c, a);
        case 3: return launch_trace_ahead<STATS, ORDERED, 3>(c, a);
        case 4: return launch_trace_ahead<STATS, ORDERED, 4>(c, a);
        default: return launch_trace_ahead<STATS, ORDERED, 1>(c, a);
    }
}

template <int N, bool STATS, bool ORDERED, int LDS_DEPTH, bool ALIKE>
int launch_trace_wide_kernel(Context* c, const TraceArgs& a) {
    static int occ = 0;
    if (occ == 0) {
        int q = 0;
        HX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&q, k_trace_wide<N, STATS, ORDERED, LDS_DEPTH, ALIKE>, kTraceBlock,
                                                             0));
        occ = std::max(q, 1);
    }
    TraceArgs t = a;
    const unsigned blocks = trace_shape(c, occ, false, t);
    hipLaunchKernelGGL((k_trace_wide<N, STATS, ORDERED, LDS_DEPTH, ALIKE>), dim3(blocks), dim3(kTraceBlock), 0, c->stream, t);
    return check_launch("trace_wide");
}

template <int N, bool STATS, bool ORDERED, int LDS_DEPTH>
int launch_trace_wide_t(Context* c, const TraceArgs& a) {
    if (!STATS && alike_pays(c, a, true)) return launch_trace_wide_kernel<N, false, ORDERED, LDS_DEPTH, true>(c, a);
    return launch_trace_wide_kernel<N, STATS, ORDERED, LDS_DEPTH, false>(c, a);
}

template <int N, bool STATS, bool ORDERED>
int launch_trace_wide_depth(Context* c, const TraceArgs& a) {
    switch (c->tune.trace_lds_stack) {
        case 0: return launch_trace_wide_t<N, STATS, ORDERED, 0>(c, a);
        case 16: return launch_trace_wide_t<N, STATS, ORDERED, 16>(c, a);
        case 24: return launch_trace_wide_t<N, STATS, ORDERED, 24>(c, a);
        case 32: return launch_trace_wide_t<N, STATS, ORDERED, 32>(c, a);
        default: return launch_trace_wide_t<N, STATS, ORDERED, 64>(c, a);
    }
}

template <int N>
int launch_trace_wide_n(Context* c, const TraceArgs& a) {
    if (a.stats)
        return a.order ? launch_trace_wide_depth<N, true, true>(c, a) : launch_trace_wide_depth<N, true, false>(c, a);
    return a.order ? launch_trace_wide_depth<N, false, true>(c, a) : launch_trace_wide_depth<N, false, false>(c, a);
}

}  // namespace

int launch_trace_wide(Context* c, int N, const TraceArgs& a) {
    if (a.n_rays <= 0) return HX_OK;
    HX_TRY(zero_control(c, a, true));
    LaunchScope ls(c, a.order ? "trace_wide_sorted" : "trace_wide");
    if (N == 4) return launch_trace_wide_n<4>(c, a);
    if (N == 8) return launch_trace_wide_n<8>(c, a);
    set_error("wide trace: %d children per node is not supported (4 or 8)", N);
    return HX_ERR_INVALID_ARG;
}

int launch_trace(Context* c, const TraceArgs& a) {
    if (a.n_rays <= 0) return HX_OK;
    HX_TRY(zero_control(c, a, false));
    LaunchScope ls(c, a.order ? "trace_sorted" : "trace");
    if (a.stats)
        return a.order ? launch_trace_postpone<true, true>(c, a) : launch_trace_postpone<true, false>(c, a);
    return a.order ? launch_trace_postpone<false, true>(c, a) : launch_trace_postpone<false, false>(c, a);
}

int launch_ray_keys(Context* c, const float4* rays, int64_t n, int method, int bits, float ray_length,
                    uint64_t* keys) {
    if (n <= 0) return HX_OK;
    LaunchScope ls(c, "ray_keys");
    const unsigned g = (unsigned)((n + 255) / 256);
    if (method == HX_RAYKEY_AILA)
        hipLaunchKernelGGL(k_ray_keys_aila, dim3(g), dim3(256), 0, c->stream, rays, n, bits, keys);
    else
        hipLaunchKernelGGL(k_ray_keys_twopoint, dim3(g), dim3(256), 0, c->stream, rays, n, bits, ray_length, keys);
    return check_launch("ray_keys");
}

}  // namespace hx
