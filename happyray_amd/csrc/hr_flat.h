// hr_flat.h -- the flat per-lane traversal state (one unit of work per step:
// a triangle test or a DDA advance) shared by the persistent kernels
// (hr_persist.hip) and the wave-cooperative trace of the path tracer
// (hr_trace.hip), and the wave-batched candidate tests both use.
//
// The operations on each ray, and their order, are those of the reference
// traversal (src/RT/Algorithm/TLGridTraverser.h:132-350, UGridTraverser.h:
// 44-177, RayTriangleIntersector.h:52-90), so every kernel built on them
// returns the one-ray-per-lane kernels' results bit for bit.
#pragma once

#include "hr_traverse.h"

namespace hr {
namespace trav {

constexpr float kInf = __builtin_huge_valf();

struct RayState {
    f3 org, dir, rcp;
    float t, tterm;
    uint32_t best;
    int cx, cy, cz;     // two-level: top cell; uniform: steps left to the grid's far side per axis (or the cell)
    float tx, ty, tz, tentry;
    uint32_t li;        // current leaf (two-level) or cell (uniform)
    int sy, sz;         // its step along y and z (x: one), with the ray's direction
    uint32_t rem;       // leaf steps left in the top cell, see kRemGuard
    float ux, uy, uz;
    float ddx, ddy, ddz;
    uint32_t it, end;   // candidate range still to test
    uint32_t pn;        // the primitive id at it, loaded one test ahead
    bool in_leaf;
};

// The leaf steps left before the ray leaves its top cell, one field per axis
// in one register: field = guard bit + (steps left - 1), so a step subtracts
// the axis' unit and the ray has left the cell when a guard bit is borrowed
// away.  A leaf resolution is at most 255, so eight bits hold the count.
constexpr uint32_t kRemX = 1u, kRemY = 1u << 9, kRemZ = 1u << 18;
constexpr uint32_t kRemGuard = (kRemX | kRemY | kRemZ) << 8;

// index of a cell; the multiplies take the 24-bit form (full rate) where the
// grid allows it, which is the same for the whole launch
__device__ __forceinline__ uint32_t cell_index(const GridRegs& G, int cx, int cy, int cz)
{
    if (G.small) {
        const uint32_t row = __umul24((uint32_t)cz, (uint32_t)G.ry) + (uint32_t)cy;
        return __umul24(row, (uint32_t)G.rx) + (uint32_t)cx;
    }
    return (uint32_t)cx + (uint32_t)cy * (uint32_t)G.rx + (uint32_t)cz * ((uint32_t)G.rx * (uint32_t)G.ry);
}

// min_dim as two masks: along x, along y, else along z
struct Axis {
    bool x, y;
};
__device__ __forceinline__ Axis min_axis(float x, float y, float z)
{
    Axis a;
    a.x = x < y && x < z;
    a.y = !(x < y) && y < z;
    return a;
}

__device__ __forceinline__ float pick(Axis a, float x, float y, float z) { return a.x ? x : (a.y ? y : z); }
__device__ __forceinline__ int pick(Axis a, int x, int y, int z) { return a.x ? x : (a.y ? y : z); }
__device__ __forceinline__ uint32_t pick(Axis a, uint32_t x, uint32_t y, uint32_t z)
{
    return a.x ? x : (a.y ? y : z);
}

template <class T>
__device__ __forceinline__ void put(Axis a, T v, T& x, T& y, T& z)
{
    x = a.x ? v : x;
    y = a.y ? v : y;
    z = (a.x || a.y) ? z : v;
}

__device__ __forceinline__ void leaf_load(const TraceScene& S, RayState& r, Work& wk)
{
    ++wk.steps;
    const uint2 leaf = S.leaves[r.li];
    r.it = leaf.x;
    r.end = leaf.y;
    if (r.it < r.end) r.pn = S.prims[r.it];
}

// visit the current top cell: non-empty cells start their leaf DDA at
// tentry (TLGridTraverser.h:147-197) and load the first leaf range.  dir is
// the ray's 1 / rcp.  The visit's six divisions are tentry / rcp, which has
// dir as the reciprocal of its divisor, and three reciprocals: in the ranges
// where the short forms are correctly rounded they take those (24 instructions
// against 66), else the divisions.
__device__ __forceinline__ void top_visit(const GridRegs& G, const TraceScene& S, RayState& r, f3 org, f3 dir,
                                          Work& wk)
{
    ++wk.steps;
    const uint2 cell = S.cells[cell_index(G, r.cx, r.cy, r.cz)];
    r.it = r.end = 0u;
    r.in_leaf = false;
    if (!(cell.y & 0x40000000u)) return;
    const int r0 = (int)(cell.y & 0xFFu), r1 = (int)((cell.y >> 8) & 0xFFu), r2 = (int)((cell.y >> 16) & 0xFFu);
    const f3 cres = mk((float)r0, (float)r1, (float)r2);
    const f3 srcp = G.csr * cres;
    const float te = r.tentry;
    f3 q = mk(div_by_rcp(te, r.rcp.x, dir.x), div_by_rcp(te, r.rcp.y, dir.y), div_by_rcp(te, r.rcp.z, dir.z));
    f3 sc = mk(rcp_in_range(srcp.x), rcp_in_range(srcp.y), rcp_in_range(srcp.z));
    {
        const f3 a = vabs(r.rcp);
        const float lo = fminf(fminf(a.x, a.y), a.z), hi = fmaxf(fmaxf(a.x, a.y), a.z);
        const float slo = fminf(fminf(srcp.x, srcp.y), srcp.z), shi = fmaxf(fmaxf(srcp.x, srcp.y), srcp.z);
        // a NaN in rcp needs no look: fminf drops it, and the quotients are NaN either way
        const bool in = lo >= kDivLow && hi <= kDivHigh && (te == 0.f || (te >= kDivLow && te <= kDivHigh)) &&
                        slo >= kRcpLow && shi <= kRcpHigh;
        if (!in) {
            q = rep(te) / r.rcp;
            sc = mk(1.f / srcp.x, 1.f / srcp.y, 1.f / srcp.z);
        }
    }
    const f3 ep = org + q;
    f3 mb;
    mb.x = (float)r.cx * G.cs.x + G.bmin.x;
    mb.y = (float)r.cy * G.cs.y + G.bmin.y;
    mb.z = (float)r.cz * G.cs.z + G.bmin.z;
    f3 cf;
    cf.x = floorf((ep - mb).x * srcp.x);
    cf.y = floorf((ep - mb).y * srcp.y);
    cf.z = floorf((ep - mb).z * srcp.z);
    cf = vmin(cres - rep(1.f), vmax(cf, rep(0.f)));
    const bool px = r.rcp.x > 0.f, py = r.rcp.y > 0.f, pz = r.rcp.z > 0.f;
    r.ux = ((cf.x + (px ? 1.f : 0.f)) * sc.x + mb.x - org.x) * r.rcp.x;
    r.uy = ((cf.y + (py ? 1.f : 0.f)) * sc.y + mb.y - org.y) * r.rcp.y;
    r.uz = ((cf.z + (pz ? 1.f : 0.f)) * sc.z + mb.z - org.z) * r.rcp.z;
    const int lx = (int)cf.x, ly = (int)cf.y, lz = (int)cf.z;
    const int r01 = r0 * r1;
    r.ddx = sc.x * fabsf(r.rcp.x);
    r.ddy = sc.y * fabsf(r.rcp.y);
    r.ddz = sc.z * fabsf(r.rcp.z);
    r.li = cell.x + (uint32_t)lx + (uint32_t)__mul24(r0, ly) + (uint32_t)__mul24(r01, lz);
    r.sy = py ? r0 : -r0;
    r.sz = pz ? r01 : -r01;
    r.rem = kRemGuard + (uint32_t)(px ? r0 - 1 - lx : lx) + (uint32_t)(py ? r1 - 1 - ly : ly) * kRemY +
            (uint32_t)(pz ? r2 - 1 - lz : lz) * kRemZ;
    r.in_leaf = true;
    leaf_load(S, r, wk);
}

__device__ __forceinline__ void uniform_load(const TraceScene& S, RayState& r, Work& wk)
{
    ++wk.steps;
    const uint2 cell = S.cells[r.li];
    r.it = cell.x;
    r.end = cell.y;
    if (r.it < r.end) r.pn = S.prims[r.it];
}

// MollerTrumboreIntersectionTest (RayTriangleIntersector.h:52-90): the hit
// distance, or +inf when the triangle is missed (barycentrics outside, or
// not beyond the intersection epsilon); a NaN distance compares false too.
// kShort: the determinant's reciprocal in its short form, for tests at full width;
// where lanes test their own candidates its check and branch cost more than the
// division (2M occlusion rays 1.45 against 1.37 ms)
template <bool kShort = true>
__device__ __forceinline__ float mt_dist(f3 org, f3 dir, f3 v0, f3 v1, f3 v2)
{
    const f3 e1 = v1 - v0;
    const f3 e2 = v2 - v0;
    const f3 pv = cross(dir, e2);
    const float det = dot(e1, pv);
    const float det_rcp = kShort ? rcp_rn(det) : 1.f / det;
    f3 tv = org - v0;
    const float alpha = det_rcp * dot(tv, pv);
    tv = cross(tv, e1);
    const float beta = det_rcp * dot(tv, dir);
    const float dist = det_rcp * dot(e2, tv);
    return (alpha >= 0.f && beta >= 0.f && alpha + beta <= 1.f && dist > kIsectEps) ? dist : kInf;
}

// one ray/triangle test; true when an any-hit ray is finished.  kMixed: the
// ray's kind is its own -- any hit when tterm > 0 (it stops once t < tterm),
// closest hit when tterm = 0 -- for kernels that trace both kinds
template <bool kAny, bool kMixed = false>
__device__ __forceinline__ bool test_one(const TraceScene& S, RayState& r, Work& wk)
{
    ++wk.tests;
    const uint32_t p = r.pn;
    ++r.it;
    // the next candidate's id is fetched while this triangle is loaded and tested
    if (r.it < r.end) r.pn = S.prims[r.it];
    f3 v0, v1, v2;
    load_tri(S.rec, p, v0, v1, v2);
    const float dist = mt_dist<false>(r.org, r.dir, v0, v1, v2);
    if (dist < r.t) {
        r.t = dist;
        r.best = p;
        return kMixed ? r.t < r.tterm : kAny;
    }
    return false;
}

// The grid steps choose the axis by selects and not by three branches: the
// lanes of a wave step along different axes, so a branch runs all three sides.

// the same step on the cell's coordinates, for kernels whose lanes test their own
// candidates: there a running index and its steps are three registers too many
// (300,000 occlusion rays 995 against 945 us)
template <bool kAny>
__device__ __forceinline__ bool advance_uniform_cells(const GridRegs& G, const TraceScene& S, RayState& r, Work& wk)
{
    const int d = min_dim(r.tx, r.ty, r.tz);
    if (kAny && r.t < r.tterm) return false;
    bool flag;
    if (d == 0) {
        flag = r.t > r.tx;
        r.cx += r.rcp.x > 0.f ? 1 : -1;
        r.tx += G.cs.x * fabsf(r.rcp.x);
        flag = flag && r.cx < G.rx && r.cx > -1;
    } else if (d == 1) {
        flag = r.t > r.ty;
        r.cy += r.rcp.y > 0.f ? 1 : -1;
        r.ty += G.cs.y * fabsf(r.rcp.y);
        flag = flag && r.cy < G.ry && r.cy > -1;
    } else {
        flag = r.t > r.tz;
        r.cz += r.rcp.z > 0.f ? 1 : -1;
        r.tz += G.cs.z * fabsf(r.rcp.z);
        flag = flag && r.cz < G.rz && r.cz > -1;
    }
    if (!flag) return false;
    r.li = cell_index(G, r.cx, r.cy, r.cz);
    uniform_load(S, r, wk);
    return true;
}

// the step after a cell's candidates are exhausted; false when the ray ends
template <bool kAny, bool kMixed = false>
__device__ __forceinline__ bool advance_uniform(const GridRegs& G, const TraceScene& S, RayState& r, Work& wk)
{
    const Axis a = min_axis(r.tx, r.ty, r.tz);
    if ((kAny || kMixed) && r.t < r.tterm) return false;
    const float tc = pick(a, r.tx, r.ty, r.tz);
    const int left = pick(a, r.cx, r.cy, r.cz) - 1;
    if (!(r.t > tc) || left == 0) return false;
    const float tn = tc + pick(a, G.cs.x, G.cs.y, G.cs.z) * fabsf(pick(a, r.rcp.x, r.rcp.y, r.rcp.z));
    put(a, tn, r.tx, r.ty, r.tz);
    put(a, left, r.cx, r.cy, r.cz);
    r.li += (uint32_t)pick(a, r.rcp.x > 0.f ? 1 : -1, r.sy, r.sz);
    uniform_load(S, r, wk);
    return true;
}

// the leaf part of a two-level advance (TLGridTraverser.h:209-286): 0 = the
// ray has ended, 1 = it moved to the next leaf of its top cell (loaded),
// 2 = it left the top cell's leaves (the top-level step comes next)
template <bool kAny, bool kMixed = false>
__device__ __forceinline__ int leaf_step(const TraceScene& S, RayState& r, Work& wk)
{
    if ((kAny || kMixed) && r.t < r.tterm) return 0;
    const Axis a = min_axis(r.ux, r.uy, r.uz);
    const float u = pick(a, r.ux, r.uy, r.uz);
    if (r.t < u) return 0;
    r.rem -= pick(a, kRemX, kRemY, kRemZ);
    if ((r.rem & kRemGuard) != kRemGuard) {
        r.in_leaf = false;
        return 2;
    }
    const float un = u + pick(a, r.ddx, r.ddy, r.ddz);
    put(a, un, r.ux, r.uy, r.uz);
    r.li += (uint32_t)pick(a, r.rcp.x > 0.f ? 1 : -1, r.sy, r.sz);
    leaf_load(S, r, wk);
    return 1;
}

// the top-level step (TLGridTraverser.h:292-347) and the visit of the next
// top cell; false when the ray leaves the grid or its hit lies before the cell
__device__ __forceinline__ bool top_step(const GridRegs& G, const TraceScene& S, RayState& r, f3 org, f3 dir,
                                         Work& wk)
{
    const Axis a = min_axis(r.tx, r.ty, r.tz);
    const float tc = pick(a, r.tx, r.ty, r.tz);
    const float rc = pick(a, r.rcp.x, r.rcp.y, r.rcp.z);
    const int c = pick(a, r.cx, r.cy, r.cz) + (rc > 0.f ? 1 : -1);
    if (!(r.t > tc) || c == pick(a, G.rx, G.ry, G.rz) || c == -1) return false;
    r.tentry = tc;
    put(a, c, r.cx, r.cy, r.cz);
    const float tn = tc + pick(a, G.cs.x, G.cs.y, G.cs.z) * fabsf(rc);
    put(a, tn, r.tx, r.ty, r.tz);
    top_visit(G, S, r, org, dir, wk);
    return true;
}

__device__ __forceinline__ bool top_step(const GridRegs& G, const TraceScene& S, RayState& r, Work& wk)
{
    return top_step(G, S, r, r.org, r.dir, wk);
}

template <bool kAny, bool kMixed = false>
__device__ __forceinline__ bool advance_two_level(const GridRegs& G, const TraceScene& S, RayState& r,
                                                  Work& wk)
{
    if (r.in_leaf) {
        const int k = leaf_step<kAny, kMixed>(S, r, wk);
        if (k != 2) return k == 1;
    }
    return top_step(G, S, r, wk);
}

// set up the DDA of a generated ray; false when it does not enter the grid.
// kCells: for advance_uniform_cells
template <bool kTwo, bool kAny, bool kMixed = false, bool kCells = false>
__device__ __forceinline__ bool ray_begin(const GridRegs& G, const TraceScene& S, RayState& r, Work& wk)
{
    r.best = S.nt;
    r.it = r.end = 0u;
    r.in_leaf = false;
    bool flag = !((kAny || kMixed) && r.t < r.tterm);
    flag = dda_setup<!kTwo>(G, r.org, r.rcp, r.tentry, r.cx, r.cy, r.cz, r.tx, r.ty, r.tz) && flag;
    if (!flag) return false;
    if (kTwo) {
        top_visit(G, S, r, r.org, r.dir, wk);
    } else {
        r.li = cell_index(G, r.cx, r.cy, r.cz);
        if (!kCells) {
            const int rxy = (int)((uint32_t)G.rx * (uint32_t)G.ry);
            r.sy = r.rcp.y > 0.f ? G.rx : -G.rx;
            r.sz = r.rcp.z > 0.f ? rxy : (int)(0u - (uint32_t)rxy);
            r.cx = r.rcp.x > 0.f ? G.rx - r.cx : r.cx + 1;
            r.cy = r.rcp.y > 0.f ? G.ry - r.cy : r.cy + 1;
            r.cz = r.rcp.z > 0.f ? G.rz - r.cz : r.cz + 1;
        }
        uniform_load(S, r, wk);
    }
    return true;
}

__device__ __forceinline__ void set_ray(RayState& r, f3 org, f3 d)
{
    r.org = org;
    r.rcp = mk(rcp_rn(d.x), rcp_rn(d.y), rcp_rn(d.z));
    r.dir = mk(rcp_rn(r.rcp.x), rcp_rn(r.rcp.y), rcp_rn(r.rcp.z));
}

// Wave-batched candidate tests.  In k_persist a lane tests its own candidates
// one per iteration, so the test code runs for the lanes that happen to have
// one -- about a third of the wave.  Here each lane hands up to kK candidates
// of its current cell or leaf to the wave per iteration; the wave tests all of
// them at full width (item k of the wave's list on lane k mod 64), each item
// reading its ray from LDS, and every hit is folded into its ray's 64-bit key
// in LDS by an atomic minimum:
//   closest hit: key = (distance bits, candidate index) -- the smallest
//     distance, the first candidate in leaf order among equal distances,
//     which is what the sequential test with `dist < t` keeps;
//   any hit: key = (candidate index, distance bits) -- the first hit in
//     leaf order, where the sequential test stops.
// Candidates are consumed in leaf order, kK at a time, so every ray ends with
// the t and primitive of the one-ray-per-lane traversal.  The ray origins and
// directions live in LDS only (the lane keeps the DDA state), which pays for
// the registers of the batched test.  An any-hit ray may test up to kK - 1
// candidates past its first hit; the work statistics count the tests of the
// sequential traversal (up to and including that hit), as the reference's
// traversal would make them.
//
// A lane also takes up to `steps_max` grid steps per iteration when the leaves
// or cells it steps into are empty, so that more lanes reach candidates by the
// wave's test batch.
//
// These kernels are bound by VALU issue under divergence (83 % busy at 48 % of
// the lanes on the 1M-triangle AO frame; 81 % at 38 % before the following), so
// what counts is instructions per iteration.  An item's owner is found without a list of items: a lane writes its number
// at its first item's place in 64 words of LDS, and a maximum scan over the
// wave carries it to the lane's other items (the owners increase with the
// items); the item's candidate is its place plus its owner's offset.  One LDS
// write per lane where a list takes two per candidate, and a quarter of its LDS.
// With the steps by selects, leaf indices kept as a running offset (no
// multiplies) and the short reciprocals: AO kernel of that frame 2.29 -> 2.12
// ms, heightfield 1024x768 camera rays 0.54 -> 0.42 and paths 0.85 -> 0.68 ms,
// 250,000 paths on a uniform grid 1.45 -> 1.17 ms.  4M rays in random order on
// 102,400 triangles stay at 1.5 ms: lines from beyond the L2 bound them (7.5 GB a
// launch at 5.8 TB/s), not the VALU.
constexpr int kBatchK = 12;   // candidates a lane hands to its wave per iteration

// Rays per wave of a launch of n rays that should spread over `blocks`
// workgroups of four waves: 64, or fewer where 64 would leave some of them
// empty.  The wave's other lanes take part in the tests only.  The time of a
// small launch is the latency of its longest rays, and an iteration is shorter
// with fewer rays in a wave (fewer kinds of steps and rounds of tests).
inline uint32_t wave_lanes(size_t n, uint32_t blocks)
{
    const size_t waves = 4 * (size_t)blocks, per = (n + waves - 1) / waves;
    return per < 1 ? 1u : (per > (size_t)kWave ? (uint32_t)kWave : (uint32_t)per);
}

inline uint32_t wave_blocks(size_t n, uint32_t lanes) { return (uint32_t)((n + 4 * (size_t)lanes - 1) / (4 * (size_t)lanes)); }

inline uint32_t device_cus()
{
    static uint32_t cached = 0;
    if (!cached) {
        int dev = 0, cus = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        cached = cus > 0 ? (uint32_t)cus : 256u;
    }
    return cached;
}

struct WaveTests {
    float4 o[kWave];          // a lane's ray: origin and current distance
    float4 d[kWave];          // direction, and (as bits) candidate - item of its run
    unsigned long long key[kWave];
    uint32_t mark[kWave];

    __device__ __forceinline__ void set_ray(uint32_t lane, f3 org, f3 dir, float t)
    {
        o[lane] = make_float4(org.x, org.y, org.z, t);
        d[lane] = make_float4(dir.x, dir.y, dir.z, 0.f);
    }
    __device__ __forceinline__ f3 org(uint32_t lane) const { return mk(o[lane].x, o[lane].y, o[lane].z); }
    __device__ __forceinline__ f3 dir(uint32_t lane) const { return mk(d[lane].x, d[lane].y, d[lane].z); }
};

// The wave's test batch over candidate references [it, end) of prims: each
// lane for which `want` holds and that has candidates left hands up to kK of
// them to the wave, the wave tests them all (each against its owner's ray in
// W) and every such lane takes its ray's result into t / best and moves it
// past the candidates.  t must be the distance in W.  Returns true on a lane
// whose any-hit ray was hit.  Every lane of the wave calls it together.  kOwn:
// the lanes' rays belong to scenes with references and records of their own;
// an item reads its owner's from own_rec / own_prims (the wave's 64 entries in
// LDS), and rec / prims are the calling lane's.
template <bool kAny, int kK, bool kOwn = false>
__device__ __forceinline__ bool wave_test_range(const float4* __restrict__ rec, const uint32_t* __restrict__ prims,
                                                WaveTests& W, uint32_t& it, uint32_t end, float& t,
                                                uint32_t& best, uint32_t lane, bool want, Work& wk,
                                                const float4* const* own_rec = nullptr,
                                                const uint32_t* const* own_prims = nullptr)
{
    bool hit = false;
    uint32_t cnt = 0;
    if (want && it < end) cnt = end - it < (uint32_t)kK ? end - it : (uint32_t)kK;
    const uint32_t incl = wave_incl_scan(cnt);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    if (total) {
        const uint32_t ex = incl - cnt;
        if (cnt) {
            W.d[lane].w = __uint_as_float(it - ex);
            W.key[lane] = ~0ull;
        }
        for (uint32_t b0 = 0; b0 < total; b0 += kWave) {
            W.mark[lane] = 0u;
            wave_sync();
            if (cnt && ex < b0 + kWave && incl > b0) W.mark[ex > b0 ? ex - b0 : 0u] = lane;
            wave_sync();
            const uint32_t o = wave_incl_max(W.mark[lane]);
            const uint32_t k = b0 + lane;
            if (k < total) {
                const float4 ro = W.o[o], rd = W.d[o];
                const uint32_t ci = k + __float_as_uint(rd.w);
                f3 v0, v1, v2;
                if (kOwn) load_tri(own_rec[o], own_prims[o][ci], v0, v1, v2);
                else load_tri(rec, prims[ci], v0, v1, v2);
                const float dist = mt_dist(mk(ro.x, ro.y, ro.z), mk(rd.x, rd.y, rd.z), v0, v1, v2);
                if (dist < ro.w) {
                    const unsigned long long db = __float_as_uint(dist);
                    atomicMin(&W.key[o], kAny ? ((unsigned long long)ci << 32 | db) : (db << 32 | ci));
                }
            }
            wave_sync();
        }
        if (cnt) {
            const unsigned long long key = W.key[lane];
            uint32_t tested = cnt;
            if (key != ~0ull) {
                const uint32_t ci = kAny ? (uint32_t)(key >> 32) : (uint32_t)key;
                t = __uint_as_float(kAny ? (uint32_t)key : (uint32_t)(key >> 32));
                best = prims[ci];
                if (kAny) {
                    hit = true;
                    tested = ci - it + 1;   // the sequential traversal stops here
                } else {
                    W.o[lane].w = t;
                }
            }
            wk.tests += tested;
            it += cnt;
        }
    }
    return hit;
}

template <bool kAny, int kK>
__device__ __forceinline__ bool wave_test_batch(const TraceScene& S, WaveTests& W, RayState& r, uint32_t lane,
                                                bool want, Work& wk)
{
    return wave_test_range<kAny, kK>(S.rec, S.prims, W, r.it, r.end, r.t, r.best, lane, want, wk);
}

// trace<> of one ray per active lane (RayTracingKernels.h:118-140: rcp = 1 / d,
// traverse, d' = 1 / rcp) with the wave's candidates tested in batches.  Every
// lane of the wave calls it together; an inactive lane takes part in the
// batches only.  kAny: t is both the start and the termination distance (the
// ray stops at its first hit below it).  Returns the hit primitive (S.nt on a
// miss) and d' in dir_out, as trace_ray does; steps_max grid steps per lane
// and batch.
template <bool kTwo, bool kAny, int kK>
__device__ __forceinline__ uint32_t trace_wave(const GridRegs& G, const TraceScene& S, WaveTests& W, bool active,
                                               f3 org, f3 d, float& t, f3& dir_out, uint32_t steps_max, Work& wk)
{
    const uint32_t lane = __lane_id();
    RayState r;
    bool live = false;
    if (active) {
        set_ray(r, org, d);
        r.t = t;
        r.tterm = t;
        live = ray_begin<kTwo, false>(G, S, r, wk);
        if (live) W.set_ray(lane, org, r.dir, t);
    }
    while (__ballot(live) != 0ull) {
        bool done = false;
        if (live && r.it >= r.end) {
#pragma unroll 1
            for (uint32_t m = 0; m < steps_max; ++m) {
                if (kTwo) {
                    bool top = true;
                    if (r.in_leaf) {
                        const int k = leaf_step<false>(S, r, wk);
                        if (k != 2) {
                            top = false;
                            done = k != 1;
                        }
                    }
                    if (top) done = !top_step(G, S, r, org, r.dir, wk);
                } else {
                    done = !advance_uniform<false>(G, S, r, wk);
                }
                if (done || r.it < r.end) break;
            }
        }
        if (wave_test_batch<kAny, kK>(S, W, r, lane, live && !done, wk)) done = true;
        if (live && done) live = false;
    }
    if (!active) return S.nt;
    t = r.t;
    dir_out = r.dir;
    return r.best;
}

}  // namespace trav
}  // namespace hr
