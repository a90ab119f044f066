// hx_presplit.hip -- budgeted triangle presplitting on gfx950.
//
// Reference (src/hippie/rt/bvh/): Presplitter.cpp:124-326 (priorities, the
// bisection for D, split tasks), PresplitterKernels.cu:11-419 (the kernels).
// In the reference this GPU variant is compiled out in favour of a CPU SBVH
// (Presplitter.cpp:11); here it is the presplitter.
//
//   priority  per triangle, (2^i (A_box - A_ideal))^(1/3) with i from the
//             highest differing bit of the 63-bit codes of its box corners;
//   D         the largest multiplier (6 bisection rounds) whose rounded budget
//             sum floor(D p) stays within beta * n;
//   split     each triangle becomes floor(D p) + 1 references by recursive
//             clipping at Morton-grid planes.
//
// Determinism: the reference appends references and tasks with atomics, so
// the reference order depends on timing.  Here a triangle's references take
// the slots [o_t, o_t + c_t] (o from a scan of c + 1), and every split hands
// its left child the first lc + 1 slots of its range, so each reference's
// slot is fixed by the split tree alone, whatever order the tasks run in.
// The float sum of the priorities (truncated to int by the reference) is an
// exact 2^-32 fixed-point sum here, and the rounded sums are 64-bit integers.
//
// Batches: with a mesh per triangle, every mesh is presplit as if alone -- its
// own box frames the codes, its own budget beta * n_m and multiplier D_m --
// and the bisection runs for all meshes at once (per-mesh sums each round).
#include <algorithm>
#include <vector>

#include "hx_device.h"
#include "hx_internal.h"

namespace hx {

namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kItems = kPsTile / kBlock;
constexpr int kTile = kPsTile;

inline unsigned grid_for(int64_t n, int block = kBlock) { return (unsigned)((n + block - 1) / block); }

struct Sum {
    HX_DEV int operator()(int a, int b) const { return a + b; }
};

// x^y in double precision from the textbook series (the host oracle runs the
// same operations): ln x = e ln2 + 2 atanh((m-1)/(m+1)) with m in
// [sqrt(1/2), sqrt(2)); e^y = 2^k e^r with |r| <= ln2/2 and the Taylor series
// of e^r.
constexpr double kLn2 = 0.69314718055994530942;
constexpr double kLn2Hi = 0.693147180369123816490;
constexpr double kLn2Lo = 1.90821492927058770002e-10;

HX_DEV double series_ln(double x) {
    int e = 0;
    double m = frexp(x, &e);
    if (m < 0.70710678118654752440) {
        m *= 2.0;
        e -= 1;
    }
    const double s = (m - 1.0) / (m + 1.0), s2 = s * s;
    double t = 1.0 / 25.0;
    for (int k = 23; k >= 1; k -= 2) t = t * s2 + 1.0 / (double)k;
    return (double)e * kLn2 + 2.0 * s * t;
}

HX_DEV double series_exp(double y) {
    const double k = rint(y / kLn2);
    const double r = (y - k * kLn2Hi) - k * kLn2Lo;
    double p = 1.0;
    for (int j = 20; j >= 1; --j) p = 1.0 + p * r / (double)j;
    return ldexp(p, (int)k);
}

HX_DEV float series_pow(float x, float y) {
    if (!(x > 0.0f) || !(x <= kMaxFloat)) return x == 0.0f ? 0.0f : x;
    return (float)series_exp((double)y * series_ln((double)x));
}

HX_DEV float ax(float3 v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }
HX_DEV void set_ax(float3& v, int a, float f) {
    if (a == 0) v.x = f;
    else if (a == 1) v.y = f;
    else v.z = f;
}
HX_DEV int ax_i(int3 v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }

// 21 bits per axis, axis 0 in bit 0 (PresplitterKernels.cu:44-55).
HX_DEV uint64_t code63(int3 q) {
    uint64_t c = 0;
#pragma unroll
    for (int i = 0; i < 21; ++i) {
        c |= (uint64_t)((q.x >> i) & 1) << (3 * i + 0);
        c |= (uint64_t)((q.y >> i) & 1) << (3 * i + 1);
        c |= (uint64_t)((q.z >> i) & 1) << (3 * i + 2);
    }
    return c;
}

HX_DEV int diff_bit(uint64_t a, uint64_t b) {
    const uint64_t d = a ^ b;
    return d ? 63 - __clzll((long long)d) : -1;
}

struct SceneFrame {
    float3 mn, dg, scale;
};

HX_DEV SceneFrame frame_of(const float* sb) {
    SceneFrame s;
    s.mn = make_float3(sb[0], sb[1], sb[2]);
    s.dg = make_float3(sb[3] - sb[0], sb[4] - sb[1], sb[5] - sb[2]);
    s.scale = make_float3(1.0f / s.dg.x, 1.0f / s.dg.y, 1.0f / s.dg.z);
    return s;
}

HX_DEV void tri_verts(const PsArgs& a, int t, float3 v[3]) {
    const int32_t* tr = a.tris + 3 * (int64_t)t;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float* p = a.verts + 3 * (int64_t)tr[k];
        v[k] = make_float3(p[0], p[1], p[2]);
    }
}

HX_DEV Box3 tri_bounds(const float3 v[3]) {
    Box3 b = box_empty();
    box_grow(b, v[0]);
    box_grow(b, v[1]);
    box_grow(b, v[2]);
    return b;
}

HX_DEV int mesh_at(const PsArgs& a, int t) { return a.mesh_of ? a.mesh_of[t] : 0; }
HX_DEV const float* frame_box(const PsArgs& a, int m) { return a.mesh_of ? a.mesh_box + 6 * (int64_t)m : a.box; }

// Per-mesh sums acc[2 * m + k] accumulated by a wave over its iterations:
// while the wave's live lanes share the mesh of the running sum it grows in
// registers, and it goes out with one device-scope atomic when the mesh
// changes (device atomics on one word serialise, so a per-wave atomic over 16M
// references would take milliseconds).  Waves whose lanes span meshes add per
// lane.  At the end the waves of the workgroup join their last runs, so a
// workgroup inside one mesh costs one atomic.
struct MeshSum {
    unsigned long long* acc;
    int k;
    int m = -1;
    unsigned long long s = 0;
    HX_DEV void flush() {
        if (m >= 0 && s && lane_id() == 0) atomicAdd(acc + 2 * (int64_t)m + k, s);
        s = 0;
    }
    // The last runs of the workgroup's waves; every thread calls it.
    HX_DEV void finish() {
        __shared__ unsigned long long sums[kWavesPerBlock];
        __shared__ int meshes[kWavesPerBlock];
        if (lane_id() == 0) {
            sums[threadIdx.x / kWave] = s;
            meshes[threadIdx.x / kWave] = m;
        }
        __syncthreads();
        if (threadIdx.x != 0) return;
        for (int w = 0; w < kWavesPerBlock;) {
            const int mesh = meshes[w];
            unsigned long long v = 0;
            for (; w < kWavesPerBlock && meshes[w] == mesh; ++w) v += sums[w];
            if (mesh >= 0 && v) atomicAdd(acc + 2 * (int64_t)mesh + k, v);
        }
    }
    HX_DEV void add(bool live, int mesh, unsigned long long v) {
        const uint64_t act = ballot64(live);
        if (!act) return;
        const int m0 = __shfl(mesh, __builtin_ctzll(act), kWave);
        if (__all(!live || mesh == m0)) {
            if (!live) v = 0;
#pragma unroll
            for (int sh = 1; sh < kWave; sh <<= 1) {
                const uint32_t lo = __shfl_xor((uint32_t)v, sh, kWave);
                const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), sh, kWave);
                v += ((unsigned long long)hi << 32) | lo;
            }
            if (m0 != m) {
                flush();
                m = m0;
            }
            s += v;
        } else if (live && v) {
            atomicAdd(acc + 2 * (int64_t)mesh + k, v);
        }
    }
};

// Each workgroup of a sum takes `chunk` consecutive triangles, so that about
// kSumBlocks workgroups cover them: enough to fill the chip, few enough that
// their atomics on one word stay cheap (16,384 triangles each left 31
// workgroups for 500,009: 176 us for the priorities and 39 us for a round of
// the bisection, now 22 and 10 us).
constexpr int kSumBlocks = 512;
inline int64_t sum_chunk(int64_t n) {
    return std::max<int64_t>((n + kSumBlocks - 1) / kSumBlocks + kBlock - 1, kBlock) / kBlock * kBlock;
}

// computePriorities (:11-71).
HX_DEV float priority(const float3 v[3], const SceneFrame& S) {
    const Box3 box = tri_bounds(v);
    const int3 qmn = make_int3(f2i_sat(((box.mn.x - S.mn.x) * S.scale.x) * 2097151.9f),
                               f2i_sat(((box.mn.y - S.mn.y) * S.scale.y) * 2097151.9f),
                               f2i_sat(((box.mn.z - S.mn.z) * S.scale.z) * 2097151.9f));
    const int3 qmx = make_int3(f2i_sat(((box.mx.x - S.mn.x) * S.scale.x) * 2097151.9f),
                               f2i_sat(((box.mx.y - S.mn.y) * S.scale.y) * 2097151.9f),
                               f2i_sat(((box.mx.z - S.mn.z) * S.scale.z) * 2097151.9f));
    const int diff = diff_bit(code63(qmn), code63(qmx));
    const int i = diff / 3 - 21;
    const float3 d1 = make_float3(v[0].x - v[1].x, v[0].y - v[1].y, v[0].z - v[1].z);
    const float3 d2 = make_float3(v[0].x - v[2].x, v[0].y - v[2].y, v[0].z - v[2].z);
    const float cx = d1.y * d2.z - d1.z * d2.y, cy = d1.z * d2.x - d1.x * d2.z, cz = d1.x * d2.y - d1.y * d2.x;
    const float ideal = fabsf(cx) + fabsf(cy) + fabsf(cz);
    return series_pow(ldexpf(1.0f, i) * (box_area(box.mn, box.mx) - ideal), 1.0f / 3.0f);
}

// Priorities and their exact fixed-point sums per mesh (macc[2m]).
__global__ __launch_bounds__(kBlock) void k_ps_priority(PsArgs a, int64_t chunk) {
    MeshSum sum{a.macc, 0};
    const int64_t end = min((int64_t)(blockIdx.x + 1) * chunk, a.n);
    for (int64_t t = blockIdx.x * chunk + threadIdx.x; t < (int64_t)(blockIdx.x + 1) * chunk; t += kBlock) {
        const bool live = t < end;
        unsigned long long s = 0;
        int m = 0;
        if (live) {
            m = mesh_at(a, (int)t);
            const SceneFrame S = frame_of(frame_box(a, m));
            float3 v[3];
            tri_verts(a, (int)t, v);
            const float p = priority(v, S);
            a.prio[t] = p;
            if (p >= 0.0f && p <= 1.0e9f) s = (unsigned long long)((double)p * 4294967296.0);
        }
        sum.add(live, m, s);
    }
    sum.finish();
}

// sumPrioritiesRound (:116-148): per-mesh sums of floor(D_m p) (macc[2m+1]).
__global__ __launch_bounds__(kBlock) void k_ps_round_sum(PsArgs a, int64_t chunk) {
    MeshSum sum{a.macc, 1};
    const int64_t end = min((int64_t)(blockIdx.x + 1) * chunk, a.n);
    for (int64_t t = blockIdx.x * chunk + threadIdx.x; t < (int64_t)(blockIdx.x + 1) * chunk; t += kBlock) {
        const bool live = t < end;
        unsigned long long s = 0;
        int m = 0;
        if (live) {
            m = mesh_at(a, (int)t);
            s = (unsigned long long)(long long)f2i_sat(a.Dm[m] * a.prio[t]);
        }
        sum.add(live, m, s);
    }
    sum.finish();
}

// Per-tile sums of floor(D p) + 1.
__global__ __launch_bounds__(kBlock) void k_ps_tile_sums(PsArgs a) {
    const int64_t base = blockIdx.x * (int64_t)kTile;
    int s = 0;
    for (int k = 0; k < kItems; ++k) {
        const int64_t t = base + k * kBlock + threadIdx.x;
        if (t < a.n) s += f2i_sat(a.Dm[mesh_at(a, (int)t)] * a.prio[t]) + 1;
    }
    s = wave_sum_i32(s);
    __shared__ int ws[kWavesPerBlock];
    if (lane_id() == 0) ws[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < kWavesPerBlock; ++w) tot += ws[w];
        a.partial[blockIdx.x] = tot;
    }
}

constexpr int kScanBlock = 1024;
__global__ __launch_bounds__(kScanBlock) void k_ps_scan(int32_t* __restrict__ partial, int count,
                                                        int32_t* __restrict__ qcount) {
    __shared__ int wt[kScanBlock / kWave];
    if (threadIdx.x < 4) qcount[threadIdx.x] = 0;
    int carry = 0;
    for (int base = 0; base < count; base += kScanBlock) {
        const int t = base + threadIdx.x;
        const int v = t < count ? partial[t] : 0;
        int tot;
        const int inc = block_inclusive_scan<kScanBlock / kWave>(v, Sum(), wt, tot);
        if (t < count) partial[t] = carry + inc - v;
        carry += tot;
    }
}

HX_DEV void write_ref(const PsArgs& a, int off, int tri, const Box3& b) {
    a.ref_min[off] = make_float4(b.mn.x, b.mn.y, b.mn.z, 0.0f);
    a.ref_max[off] = make_float4(b.mx.x, b.mx.y, b.mx.z, 0.0f);
    a.ref_tri[off] = tri;
}

// Append tasks to queue q, counted in qcount[cnt] (the order of the queue does
// not matter, every task carries its output slots).  The R batches of tasks of a
// workgroup share one slot reservation: one atomic per wave on the one counter
// (~10 ns each) was most of the first pass, 63 us for 500,009 triangles, now
// 16 us.  reserve: first slot of batch r for this thread's lane, every
// thread of the workgroup calls it.
template <int R>
HX_DEV void reserve_slots(const PsArgs& a, int cnt, const bool (&live)[R], int (&slot)[R]) {
    __shared__ int s_base[R][kWavesPerBlock];
    const int w = threadIdx.x / kWave;
    uint64_t m[R];
    __syncthreads();  // the previous reservation has been read
#pragma unroll
    for (int r = 0; r < R; ++r) {
        m[r] = ballot64(live[r]);
        if (lane_id() == 0) s_base[r][w] = __popcll(m[r]);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int r = 0; r < R; ++r)
            for (int v = 0; v < kWavesPerBlock; ++v) {
                const int x = s_base[r][v];
                s_base[r][v] = tot;
                tot += x;
            }
        const int base = tot ? atomicAdd(a.qcount + cnt, tot) : 0;
        for (int r = 0; r < R; ++r)
            for (int v = 0; v < kWavesPerBlock; ++v) s_base[r][v] += base;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) slot[r] = s_base[r][w] + count_below(m[r]);
}

HX_DEV void push_task(const PsArgs& a, int q, int slot, bool live, int tri, int count, int off, const Box3& b) {
    if (!live || slot >= a.queue_cap) return;  // an overflow is reported by the host from the count
    a.task[q][slot] = make_int4(tri, count, off, 0);
    a.tmn[q][slot] = make_float4(b.mn.x, b.mn.y, b.mn.z, 0.0f);
    a.tmx[q][slot] = make_float4(b.mx.x, b.mx.y, b.mx.z, 0.0f);
}

// initSplitTasks (:150-187): slot offsets from the tile scan; an unsplit
// triangle is written as its own reference at once, the others are queued.
__global__ __launch_bounds__(kBlock) void k_ps_init(PsArgs a) {
    __shared__ int wt[kWavesPerBlock];
    const int64_t base = blockIdx.x * (int64_t)kTile;
    int carry = a.partial[blockIdx.x];
    int budget[kItems], slot[kItems];
    bool split[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int64_t t = base + k * kBlock + threadIdx.x;
        budget[k] = t < a.n ? f2i_sat(a.Dm[mesh_at(a, (int)t)] * a.prio[t]) : 0;
        split[k] = budget[k] > 0;
    }
    reserve_slots(a, 0, split, slot);
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int64_t t = base + k * kBlock + threadIdx.x;
        const bool in = t < a.n;
        const int cnt = budget[k];
        const int w = in ? cnt + 1 : 0;
        int tot;
        const int inc = block_inclusive_scan<kWavesPerBlock>(w, Sum(), wt, tot);
        const int off = carry + inc - w;
        carry += tot;
        Box3 b = box_empty();
        if (in) {
            float3 v[3];
            tri_verts(a, (int)t, v);
            b = tri_bounds(v);
            if (cnt == 0) write_ref(a, off, (int)t, b);
        }
        push_task(a, 0, slot[k], split[k], (int)t, cnt, off, b);
    }
}

// split (:189-419) of every queued task into two children; a child with no
// budget left is written as a reference, the others go to the next queue.
HX_DEV void split_task(const PsArgs& a, int q, int next, bool live, int k) {
    int tri = 0, lc = 0, rc = 0, loff = 0, roff = 0;
    Box3 lb = box_empty(), rb = box_empty();
    if (live) {
        const int4 tk = a.task[q][k];
        const float4 bmn4 = a.tmn[q][k], bmx4 = a.tmx[q][k];
        Box3 box;
        box.mn = make_float3(bmn4.x, bmn4.y, bmn4.z);
        box.mx = make_float3(bmx4.x, bmx4.y, bmx4.z);
        tri = tk.x;
        const SceneFrame S = frame_of(frame_box(a, mesh_at(a, tri)));
        const int3 qmn = make_int3(f2i_sat(((box.mn.x - S.mn.x) / S.dg.x) * 2097151.9f),
                                   f2i_sat(((box.mn.y - S.mn.y) / S.dg.y) * 2097151.9f),
                                   f2i_sat(((box.mn.z - S.mn.z) / S.dg.z) * 2097151.9f));
        const int3 qmx = make_int3(f2i_sat(((box.mx.x - S.mn.x) / S.dg.x) * 2097151.9f),
                                   f2i_sat(((box.mx.y - S.mn.y) / S.dg.y) * 2097151.9f),
                                   f2i_sat(((box.mx.z - S.mn.z) / S.dg.z) * 2097151.9f));
        const int diff = diff_bit(code63(qmn), code63(qmx));
        int axis;
        float pos;
        if (diff >= 0) {
            axis = diff % 3;
            pos = 0.0f;
            float delta = 0.5f;
            const int qa = ax_i(qmx, axis);
            for (int i = 20; i >= diff / 3; --i) {
                if ((qa >> i) & 1) pos += delta;
                delta *= 0.5f;
            }
            pos = pos * ax(S.dg, axis) + ax(S.mn, axis);
            if (ax(box.mn, axis) >= pos || ax(box.mx, axis) <= pos) pos = (ax(box.mn, axis) + ax(box.mx, axis)) * 0.5f;
        } else {
            const float dx = box.mx.x - box.mn.x, dy = box.mx.y - box.mn.y, dz = box.mx.z - box.mn.z;
            axis = (dx > dy && dx > dz) ? 0 : (dy > dz ? 1 : 2);
            pos = (ax(box.mn, axis) + ax(box.mx, axis)) * 0.5f;
        }
        float3 v[3];
        tri_verts(a, tri, v);
        // Edges (v2,v0), (v0,v1), (v1,v2): each start vertex goes to the side(s)
        // it lies on, and a crossing edge adds its plane point to both.
        int j1 = 2;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int j0 = j1;
            j1 = i;
            const float3 p0 = v[j0], p1 = v[j1];
            const float pa = ax(p0, axis), pb = ax(p1, axis);
            if (pa <= pos) box_grow(lb, p0);
            if (pa >= pos) box_grow(rb, p0);
            if ((pa < pos && pb > pos) || (pa > pos && pb < pos)) {
                const float tt = maxs(mins((pos - pa) / (pb - pa), 1.0f), 0.0f);
                const float u = 1.0f - tt;
                const float3 m = make_float3(p0.x * u + p1.x * tt, p0.y * u + p1.y * tt, p0.z * u + p1.z * tt);
                box_grow(lb, m);
                box_grow(rb, m);
            }
        }
        set_ax(lb.mx, axis, pos);
        set_ax(rb.mn, axis, pos);
        lb.mn = make_float3(maxs(lb.mn.x, box.mn.x), maxs(lb.mn.y, box.mn.y), maxs(lb.mn.z, box.mn.z));
        lb.mx = make_float3(mins(lb.mx.x, box.mx.x), mins(lb.mx.y, box.mx.y), mins(lb.mx.z, box.mx.z));
        rb.mn = make_float3(maxs(rb.mn.x, box.mn.x), maxs(rb.mn.y, box.mn.y), maxs(rb.mn.z, box.mn.z));
        rb.mx = make_float3(mins(rb.mx.x, box.mx.x), mins(rb.mx.y, box.mx.y), mins(rb.mx.z, box.mx.z));
        // AABB::longest (util/AABB.h:38) returns bool: 1 unless the box is a point.
        const float ll = fmaxf(fmaxf(lb.mx.x - lb.mn.x, lb.mx.y - lb.mn.y), lb.mx.z - lb.mn.z) != 0.0f ? 1.0f : 0.0f;
        const float rl = fmaxf(fmaxf(rb.mx.x - rb.mn.x, rb.mx.y - rb.mn.y), rb.mx.z - rb.mn.z) != 0.0f ? 1.0f : 0.0f;
        lc = f2i_sat(((float)(tk.y - 1) * ll) / (ll + rl) + 0.5f);
        rc = tk.y - 1 - lc;
        loff = tk.z;
        roff = tk.z + lc + 1;
        if (lc <= 0) write_ref(a, loff, tri, lb);
        if (rc <= 0) write_ref(a, roff, tri, rb);
    }
    const bool again[2] = {live && lc > 0, live && rc > 0};
    int slot[2];
    reserve_slots(a, next, again, slot);
    push_task(a, q ^ 1, slot[0], again[0], tri, lc, loff, lb);
    push_task(a, q ^ 1, slot[1], again[1], tri, rc, roff, rb);
}

// Split round `round`: the tasks of queue round & 1, counted in qcount[round % 3],
// into the other queue, counted in the next word; the word after that is cleared
// for the round to come, and qcount[3] keeps the largest count.  The rounds read
// their counts on the device, so the host reads one count per batch of rounds
// instead of one per round; an empty round costs a launch.
__global__ __launch_bounds__(kBlock) void k_ps_split(PsArgs a, int round) {
    const int cur = round % 3, next = (round + 1) % 3;
    const int count = a.qcount[cur];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.qcount[(round + 2) % 3] = 0;
        if (count > a.qcount[3]) a.qcount[3] = count;
    }
    const int64_t todo = min((int64_t)count, a.queue_cap);
    for (int64_t base = blockIdx.x * (int64_t)kBlock; base < todo; base += (int64_t)gridDim.x * kBlock)
        split_task(a, round & 1, next, base + threadIdx.x < todo, (int)(base + threadIdx.x));
}

__global__ void k_ps_zero_u64(unsigned long long* p, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

constexpr int kSplitBatch = 4;       // split rounds launched between host reads
constexpr int kSplitBlocks = 2048;

// computeD (Presplitter.cpp:124-155) for every mesh, Smax = (int)(beta * n_m); a
// mesh whose priority sum floors to 0 gets D = 0 (no splits).  Step 0 takes the
// priority sums and sets the first multiplier, step 1 the bounds from its
// rounded sum, steps 2..7 a bisection each; after step kBisect + 1 Dm is the
// lower bound.  Clears the sums for the next round.  On the device, the eight
// rounds run without the host (each was a round trip of 40 to 75 us).
constexpr int kBisect = 6;
__global__ __launch_bounds__(kBlock) void k_ps_bisect(PsArgs a, int M, int step) {
    const int m = blockIdx.x * kBlock + threadIdx.x;
    if (m >= M) return;
    const int64_t smax = a.smax[m];
    float dmin = a.dlim[2 * m], dmax = a.dlim[2 * m + 1];
    if (step == 0) {
        const int64_t s1 = (int64_t)(a.macc[2 * (int64_t)m] >> 32);
        a.sum1[m] = s1;
        dmin = s1 > 0 ? (float)(smax / s1) : 0.0f;
        dmax = 0.0f;
    }
    const bool live = a.sum1[m] > 0;
    const int64_t s = (int64_t)a.macc[2 * (int64_t)m + 1];
    if (step == 1) {
        dmax = live ? (dmin * (float)smax) / (float)s : 0.0f;
    } else if (step > 1 && live) {
        const float cur = 0.5f * (dmin + dmax);
        if (s > smax) dmax = cur;
        else dmin = cur;
    }
    a.dlim[2 * m] = dmin;
    a.dlim[2 * m + 1] = dmax;
    const bool bisecting = step >= 1 && step <= kBisect;
    a.Dm[m] = bisecting ? (live ? 0.5f * (dmin + dmax) : 0.0f) : dmin;
    a.macc[2 * (int64_t)m] = 0;
    a.macc[2 * (int64_t)m + 1] = 0;
}

__global__ __launch_bounds__(kBlock) void k_refs_to_tris(int32_t* __restrict__ ids, const int32_t* __restrict__ ref_tri,
                                                         int64_t n) {
    const int64_t p = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if (p < n) ids[p] = ref_tri[ids[p]];
}

}  // namespace

int launch_refs_to_tris(Context* c, int32_t* ids, const int32_t* ref_tri, int64_t n) {
    hipLaunchKernelGGL(k_refs_to_tris, dim3(grid_for(n)), dim3(kBlock), 0, c->stream, ids, ref_tri, n);
    return check_launch("refs_to_tris");
}

int launch_presplit_count(Context* c, const PsArgs& a, float beta, int M, const int64_t* tri_counts,
                          int64_t* ref_counts, float* D_out) {
    LaunchScope ls(c, "presplit_count");
    const int64_t chunk = sum_chunk(a.n);
    const dim3 blocks((unsigned)((a.n + chunk - 1) / chunk));
    std::vector<int64_t> smax(M);
    for (int m = 0; m < M; ++m) smax[m] = f2i_host(beta * (float)tri_counts[m]);
    HX_HIP(hipMemcpyAsync(a.smax, smax.data(), sizeof(int64_t) * (size_t)M, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_ps_zero_u64, dim3(std::min<unsigned>(grid_for(2 * (int64_t)M), 1024u)), dim3(kBlock), 0,
                       c->stream, a.macc, 2 * (int64_t)M);
    HX_TRY(check_launch("ps_zero"));
    hipLaunchKernelGGL(k_ps_priority, blocks, dim3(kBlock), 0, c->stream, a, chunk);
    HX_TRY(check_launch("ps_priority"));
    for (int step = 0; step <= kBisect + 1; ++step) {
        hipLaunchKernelGGL(k_ps_bisect, dim3(grid_for(M)), dim3(kBlock), 0, c->stream, a, M, step);
        HX_TRY(check_launch("ps_bisect"));
        hipLaunchKernelGGL(k_ps_round_sum, blocks, dim3(kBlock), 0, c->stream, a, chunk);
        HX_TRY(check_launch("ps_round_sum"));
    }
    std::vector<unsigned long long> h(2 * (size_t)M);
    HX_HIP(hipMemcpyAsync(h.data(), a.macc, sizeof(unsigned long long) * h.size(), hipMemcpyDeviceToHost,
                          c->stream));
    HX_HIP(hipMemcpyAsync(D_out, a.Dm, sizeof(float) * (size_t)M, hipMemcpyDeviceToHost, c->stream));
    HX_HIP(hipStreamSynchronize(c->stream));
    for (int m = 0; m < M; ++m) ref_counts[m] = tri_counts[m] + (int64_t)h[2 * (size_t)m + 1];
    return HX_OK;
}

int launch_presplit_refs(Context* c, const PsArgs& a, int64_t n_refs) {
    LaunchScope ls(c, "presplit_split");
    const int64_t n = a.n;
    const int ntiles = (int)((n + kTile - 1) / kTile);
    hipLaunchKernelGGL(k_ps_tile_sums, dim3(ntiles), dim3(kBlock), 0, c->stream, a);
    HX_TRY(check_launch("ps_tile_sums"));
    hipLaunchKernelGGL(k_ps_scan, dim3(1), dim3(kScanBlock), 0, c->stream, a.partial, ntiles, a.qcount);
    HX_TRY(check_launch("ps_scan"));
    hipLaunchKernelGGL(k_ps_init, dim3(ntiles), dim3(kBlock), 0, c->stream, a);
    HX_TRY(check_launch("ps_init"));
    // Every split consumes one unit of budget, so the rounds end; the bound
    // guards against a miscount.
    const unsigned grid = std::min<unsigned>(grid_for(a.queue_cap), kSplitBlocks);
    int32_t q[4];
    for (int round = 0;;) {
        for (int k = 0; k < kSplitBatch; ++k, ++round) {
            hipLaunchKernelGGL(k_ps_split, dim3(grid), dim3(kBlock), 0, c->stream, a, round);
            HX_TRY(check_launch("ps_split"));
        }
        HX_HIP(hipMemcpyAsync(q, a.qcount, sizeof(q), hipMemcpyDeviceToHost, c->stream));
        HX_HIP(hipStreamSynchronize(c->stream));
        const int32_t most = std::max(q[3], q[round % 3]);
        if ((int64_t)most > a.queue_cap || round > n_refs + kSplitBatch) {
            set_error("presplit: split queue overflow (%d tasks, capacity %lld)", most, (long long)a.queue_cap);
            return HX_ERR_HIP;
        }
        if (q[round % 3] == 0) return HX_OK;
    }
}

}  // namespace hx
