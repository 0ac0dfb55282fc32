// sppm_trace.h -- closest hit through the GPU-built wide BVH.
//
// Replaces N_BVH<Triangle_ID, Ray, 8>::ClosestHit (bvh8.h:568-641).  The
// triangle test is Isc::Intersect(Ray, Triangle_ID) (Intersect.cpp:67-89)
// with identical float operations; a hit is accepted when t > MinT and
// (t < best, or t == best and the facet id is lower): ties go to the lowest
// facet id, so the result is independent of the tree shape and width.
// Child boxes are padded by 0.001 like AABB::Expand (Intersect.cpp:556-575) and
// rounded outwards to the node's byte grid, and the slab test is inclusive, so no
// box containing an accepted hit is ever culled: the rounding of the slab
// distances, fma(byte, step/d, (origin - o)/d), is far below the padding
// (culling decides only which boxes are visited, never the hit).
//
// What bounds it: vector instructions, most of them issued for few lanes.  A
// path wave that traced all its lanes' rays to the end, then shaded them, ran
// with 8 of 64 lanes on average.  Hence three things.  The traversal's state can
// be left and taken up again (RayTrav), so that a wave shades the rays that are
// done while the others go on; the lanes of a wave take node steps and leaf
// steps by turns (trav_run); and a leaf's triangles are spread over the lanes
// (trav_leaves).  With the byte nodes and their one-word sort keys (about 300
// instructions and 5 loads a node; 900, with a branch per comparator, and 14)
// the photon pass alone went from 2.80 to 1.89 ms (1M photons, 203k triangles),
// 11.3 to 6.0 ms (4M photons, 500k triangles of rough glass), the eye pass
// 0.72 to 0.58 and 2.39 to 1.64 ms (1024^2), 1M rays through the 203k triangles
// 0.62 to 0.41 ms, 20k shadow rays 0.078 to 0.053 ms.  (These photon and eye
// times include the gains of the shading, see lobe_draw, and of the collapse.)
//
// Traversal descends into the nearest intersected child and pushes the
// others far-to-near.  The first TRACE_LDS stack entries of a lane live in
// LDS (entry s of lane t at lds[s * 64 + t], bank-conflict free, with its
// box's entry distance at lds[(TRACE_LDS + s) * 64 + t], so a pop skips
// boxes that lie beyond the best hit found since the push); deeper entries
// spill to a global area (entry s at glob[(s - TRACE_LDS) * gstride]), so the
// LDS footprint, and with it the occupancy, does not depend on the tree
// depth.  The host sizes the total capacity from the measured depth.
#pragma once
#include "sppm_device.h"

namespace sppm {

struct TraceStack {
    uint32_t* lds;   // LDS base + lane; stride 64 (PATH_BLOCK)
    uint32_t* glob;  // spill area + the lane's slot; stride gstride
    int gstride;
    int cap;         // total entries
    uint32_t* own;   // LDS of the wave: 32 words (trav_leaves)
};

struct HitRec {
    float t, u, v;
    int facet;  // -1: miss
    int slot;   // leaf-triangle index (sorted order)
    bool tie;   // another facet is hit at exactly the same t: the reference keeps the
                // last-tested one (bvh8.h:591), which depends on its tree; here the lowest id
};

__device__ __forceinline__ bool tri_test(const float4* __restrict__ tri, int slot, f3 org, f3 dir, float& t,
                                         float& u, float& v, int& facet) {
    float4 A = tri[3 * slot + 0];
    float4 B = tri[3 * slot + 1];
    float4 C = tri[3 * slot + 2];
    facet = __float_as_int(A.w);
    f3 p0 = mk(A.x, A.y, A.z);
    f3 e1 = mk(B.x, B.y, B.z);
    f3 e2 = mk(C.x, C.y, C.z);
    f3 ps = cross(dir, e2);
    float a = dot(e1, ps);
    if (a > -1.17549435e-38f && a < 1.17549435e-38f) return false;  // |a| < FLT_MIN
    float f = 1.0f / a;
    f3 s = org - p0;
    float uu = f * dot(s, ps);
    if (uu < 0.0f || uu > 1.0f) return false;
    f3 q = cross(s, e1);
    float vv = f * dot(dir, q);
    if (vv < 0.0f || uu + vv > 1.0f) return false;
    t = f * dot(e2, q);
    u = uu;
    v = vv;
    return true;
}

__device__ __forceinline__ void cswap(uint32_t& a, uint32_t& b) {
    const uint32_t lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}
template <int W>
__device__ __forceinline__ void sort_keys(uint32_t* k) {
    if constexpr (W == 2) {
        cswap(k[0], k[1]);
    } else if constexpr (W == 4) {
        cswap(k[0], k[1]); cswap(k[2], k[3]);
        cswap(k[0], k[2]); cswap(k[1], k[3]);
        cswap(k[1], k[2]);
    } else {
        // Batcher odd-even merge sort network for 8 inputs (19 comparators)
        cswap(k[0], k[1]); cswap(k[2], k[3]); cswap(k[4], k[5]); cswap(k[6], k[7]);
        cswap(k[0], k[2]); cswap(k[1], k[3]); cswap(k[4], k[6]); cswap(k[5], k[7]);
        cswap(k[1], k[2]); cswap(k[5], k[6]);
        cswap(k[0], k[4]); cswap(k[1], k[5]); cswap(k[2], k[6]); cswap(k[3], k[7]);
        cswap(k[2], k[4]); cswap(k[3], k[5]);
        cswap(k[1], k[2]); cswap(k[3], k[4]); cswap(k[5], k[6]);
    }
}

// The ray in the frame of a node (layout: sppm_layout.h): plane q of axis a
// is crossed at fma(q, step.a, org.a).
struct NodeFrame {
    f3 step, org;
};
__device__ __forceinline__ NodeFrame node_frame(const uint32_t* w, f3 org, f3 inv) {
    NodeFrame f;
    f.step.x = __uint_as_float((w[3] & 0x3ffu) << 21) * inv.x;
    f.step.y = __uint_as_float(((w[3] >> 10) & 0x3ffu) << 21) * inv.y;
    f.step.z = __uint_as_float((w[3] >> 20) << 21) * inv.z;
    f.org.x = (__uint_as_float(w[0]) - org.x) * inv.x;
    f.org.y = (__uint_as_float(w[1]) - org.y) * inv.y;
    f.org.z = (__uint_as_float(w[2]) - org.z) * inv.z;
    return f;
}
__device__ __forceinline__ float byte_f(uint32_t w, int k) { return (float)((w >> (8 * k)) & 0xffu); }
// The planes of axis a that a ray crosses first (far: last), child c's in byte
// c & 3 of word c >> 2; neg: the ray runs towards smaller coordinates.
template <int W>
__device__ __forceinline__ void node_planes(const uint32_t* w, int a, bool neg, uint32_t* near_, uint32_t* far_) {
    const uint32_t* p = w + NODE_PLANES(W);
    if constexpr (W == 8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t lo = p[4 * a + h], hi = p[4 * a + 2 + h];
            near_[h] = neg ? hi : lo;
            far_[h] = neg ? lo : hi;
        }
    } else if constexpr (W == 4) {
        const uint32_t lo = p[2 * a], hi = p[2 * a + 1];
        near_[0] = neg ? hi : lo;
        far_[0] = neg ? lo : hi;
    } else {
        const uint32_t lo = p[a], hi = p[a] >> 16;
        near_[0] = neg ? hi : lo;
        far_[0] = neg ? lo : hi;
    }
}
// The traversal reference of the child in a slot: m its byte, p the byte of the
// slot before (0 for the first).
__device__ __forceinline__ uint32_t node_ref(const uint32_t* w, uint32_t m, uint32_t p) {
    const uint32_t leaf = LEAF_BIT | ((w[5] + (p & 0x7fu)) << 3) | (((m & 0x7fu) - (p & 0x7fu) - 1u) & 7u);
    return m & NODE_LEAF ? leaf : w[4] + (m & 0x7fu);
}
template <int W>
__device__ __forceinline__ uint32_t node_child(const uint32_t* w, uint32_t slot) {
    if constexpr (W == 8) {
        const unsigned long long m = ((unsigned long long)w[7] << 32) | w[6];
        return node_ref(w, (uint32_t)(m >> (8u * slot)) & 0xffu, (uint32_t)((m << 8) >> (8u * slot)));
    } else {
        return node_ref(w, (w[6] >> (8u * slot)) & 0xffu, (w[6] << 8) >> (8u * slot));
    }
}

// Pops the next stack entry whose box may still hold an accepted hit: an
// LDS entry keeps its box's entry distance and is skipped once that is
// beyond best (the rule it was pushed under; a hit inside the box lies at or
// beyond it); spilled entries are always taken.  EMPTY_CHILD when none is left.
__device__ __forceinline__ uint32_t trace_pop(const TraceStack& ts, int& sp, float best) {
    while (sp > 0) {
        --sp;
        if (sp >= ts.cap) return EMPTY_CHILD;  // overflowed stack: stop (flagged)
        if (sp < TRACE_LDS) {
            // as bits: a best below zero culls nothing
            if (ts.lds[(TRACE_LDS + sp) * 64] > __float_as_uint(best)) continue;
            return ts.lds[sp * 64];
        }
        return ts.glob[(size_t)(sp - TRACE_LDS) * ts.gstride];
    }
    return EMPTY_CHILD;
}
// A closest hit in progress.  Only what cannot be formed again from the ray
// is kept, so a path kernel can hold it beside the path's state: u, v and the
// facet come from the hit triangle once the ray is done.
struct RayTrav {
    float best;    // distance of the closest hit so far (FLT_MAX: none)
    int slot;      // its leaf triangle
    uint32_t ref;  // the node or leaf range to visit next; EMPTY_CHILD: the ray is done
    int sp;        // stack entries
    bool tie;
};
__device__ __forceinline__ void trav_begin(RayTrav& R) {
    R.best = 3.40282347e38f;  // FLT_MAX = Ray::m_MaxT
    R.slot = -1;
    R.ref = 0;  // root node
    R.sp = 0;
    R.tie = false;
}

// One inner node: the hit children but the nearest are pushed far to near.
// A child is sorted by its box's entry distance with the slot in the lowest
// three bits (a distance below the true one, so culling by it stays safe);
// minima and maxima of one word instead of compared pairs, and its reference
// is formed only when it is pushed.
template <int W>
__device__ __forceinline__ void trav_node(const SceneDev& S, f3 org, f3 inv, const TraceStack& ts, RayTrav& R,
                                          uint32_t* flags) {
    constexpr int NW = node_words(W);
    uint32_t w[NW];
    const uint4* nd = reinterpret_cast<const uint4*>(S.nodes + (size_t)R.ref * NW);
#pragma unroll
    for (int k = 0; k < NW / 4; ++k) {
        const uint4 q = nd[k];
        w[4 * k] = q.x; w[4 * k + 1] = q.y; w[4 * k + 2] = q.z; w[4 * k + 3] = q.w;
    }
    const NodeFrame f = node_frame(w, org, inv);
    uint32_t nx[2], fx[2], ny[2], fy[2], nz[2], fz[2];
    node_planes<W>(w, 0, inv.x < 0.0f, nx, fx);
    node_planes<W>(w, 1, inv.y < 0.0f, ny, fy);
    node_planes<W>(w, 2, inv.z < 0.0f, nz, fz);
    uint32_t key[W];
#pragma unroll
    for (int c = 0; c < W; ++c) {
        const int h = c >> 2, b = c & 3;
        const float tn = fmaxf(fmaxf(fmaf(byte_f(nx[h], b), f.step.x, f.org.x), fmaf(byte_f(ny[h], b), f.step.y, f.org.y)),
                               fmaf(byte_f(nz[h], b), f.step.z, f.org.z));
        const float tf = fminf(fminf(fmaf(byte_f(fx[h], b), f.step.x, f.org.x), fmaf(byte_f(fy[h], b), f.step.y, f.org.y)),
                               fmaf(byte_f(fz[h], b), f.step.z, f.org.z));
        // tn <= tf: a ray of NaNs meets nothing
        const bool hit = (tn <= fminf(tf, R.best)) & (tf >= 0.0f);
        key[c] = hit ? (__float_as_uint(fmaxf(tn, 0.0f)) & ~7u) | (uint32_t)c : EMPTY_CHILD;
    }
    sort_keys<W>(key);
    if (key[0] == EMPTY_CHILD) {
        R.ref = trace_pop(ts, R.sp, R.best);
        return;
    }
#pragma unroll
    for (int c = W - 1; c >= 1; --c) {
        if (key[c] != EMPTY_CHILD) {
            const uint32_t r = node_child<W>(w, key[c] & 7u);
            if (R.sp < TRACE_LDS) {
                ts.lds[R.sp * 64] = r;
                ts.lds[(TRACE_LDS + R.sp) * 64] = key[c] & ~7u;
            }
            else if (R.sp < ts.cap) ts.glob[(size_t)(R.sp - TRACE_LDS) * ts.gstride] = r;
            else *flags |= 4u;
            ++R.sp;
        }
    }
    R.ref = node_child<W>(w, key[0] & 7u);
}

// A triangle's hit against the closest so far: nearer wins, at the same
// distance the lower facet.
__device__ __forceinline__ void trav_take(const SceneDev& S, RayTrav& R, float t, int slot, int fid, bool tied) {
    if (!(t <= R.best)) return;
    bool take = t < R.best;
    if (!take && R.slot >= 0) {
        const int bf = __float_as_int(S.tri[3 * R.slot].w);
        R.tie = R.tie || tied || fid != bf;
        take = fid < bf;
    } else {
        R.tie = tied;
    }
    if (take) {
        R.best = t;
        R.slot = slot;
    }
}

// Leaves of the wave: up to 16 of the lanes in `leaves` are served, four of
// each one's triangles at a time, one triangle per lane.  One lane testing its
// leaf's triangles in turn would keep the wave for as many dependent loads as
// the longest leaf has triangles, at six lanes of 64 on average.  own: LDS, the
// lane served by each group of four.  Called by all active lanes together; act:
// those lanes.
template <int Q>
__device__ __forceinline__ void trav_leaves(const SceneDev& S, f3 org, f3 dir, float tmin, const TraceStack& ts,
                                            unsigned long long leaves, RayTrav& R) {
    const int lane = (int)(threadIdx.x & 63u);
    const int rank = __popcll(leaves & ((1ull << lane) - 1ull));
    const bool served = ((leaves >> lane) & 1ull) != 0ull && rank < 64 / Q;
    // lane rank * Q + k tests triangle k of the leaf of the rank-th lane
    uint32_t* const own = ts.own;
    if (served) own[rank] = (uint32_t)lane;
    __builtin_amdgcn_wave_barrier();
    const int nleaf = min(__popcll(leaves), 64 / Q);
    const int g = lane / Q, k = lane % Q;
    const int src = (int)own[min(g, nleaf - 1)];
    const uint32_t ref = (uint32_t)__shfl((int)R.ref, src, 64);
    const f3 o = mk(__shfl(org.x, src, 64), __shfl(org.y, src, 64), __shfl(org.z, src, 64));
    const f3 d = mk(__shfl(dir.x, src, 64), __shfl(dir.y, src, 64), __shfl(dir.z, src, 64));
    const int cnt = (int)(ref & 7u) + 1;
    int s = (int)((ref & ~LEAF_BIT) >> 3) + min(k, cnt - 1);
    float t, u, v;
    int fid;
    if (!(tri_test(S.tri, s, o, d, t, u, v, fid) && t > tmin)) t = __int_as_float(0x7f800000);
    bool tied = false;
#pragma unroll
    for (int off = 1; off < Q; off <<= 1) {
        const float t2 = __shfl_xor(t, off, 64);
        const int f2 = __shfl_xor(fid, off, 64), s2 = __shfl_xor(s, off, 64);
        const bool ti2 = __shfl_xor((int)tied, off, 64) != 0;
        const bool eq = t2 == t, sw = t2 < t || (eq && f2 < fid);
        tied = eq ? (tied || ti2 || f2 != fid) : (sw ? ti2 : tied);
        t = sw ? t2 : t;
        fid = sw ? f2 : fid;
        s = sw ? s2 : s;
    }
    // back to the ray's lane
    const int from = (rank * Q) & 63;
    const float rt = __shfl(t, from, 64);
    const int rf = __shfl(fid, from, 64), rs = __shfl(s, from, 64), ri = __shfl((int)tied, from, 64);
    if (served) {
        if (rt < __int_as_float(0x7f800000)) trav_take(S, R, rt, rs, rf, ri != 0);
        // the leaf's other triangles, if any
        R.ref = (R.ref & 7u) >= (uint32_t)Q ? R.ref + 8u * Q - Q : trace_pop(ts, R.sp, R.best);
    }
}

// The triangles of a lane's own leaf.
__device__ __forceinline__ void trav_leaf(const SceneDev& S, f3 org, f3 dir, float tmin, const TraceStack& ts,
                                          RayTrav& R) {
    const int s0 = (int)((R.ref & ~LEAF_BIT) >> 3), s1 = s0 + (int)(R.ref & 7u);
    for (int s = s0; s <= s1; ++s) {
        float t, u, v;
        int fid;
        if (tri_test(S.tri, s, org, dir, t, u, v, fid) && t > tmin) trav_take(S, R, t, s, fid, false);
    }
    R.ref = trace_pop(ts, R.sp, R.best);
}

// Runs the wave's rays (lanes whose ref is not EMPTY_CHILD) until at most
// `stop` of them are left.  A step is either an inner node for the lanes that
// stand at one or leaves for the others, whichever more lanes ask for (a leaf
// step costs about two thirds of a node's, so half as many lanes are enough for
// it), so a lane at a leaf does not sit through another lane's node or the
// other way round.
// WAVE: the whole wave calls this together, and its lanes share the leaves'
// triangles; eight lanes for a leaf (all its triangles) where no more than
// eight lanes stand at one, else four.  Otherwise the lanes that call it are
// the wave, and each tests its own leaf.
constexpr int TRAV_LEAF_VOTE = 2;
template <int W, bool WAVE>
__device__ __forceinline__ void trav_run(const SceneDev& S, f3 org, f3 dir, float tmin, const TraceStack& ts, int stop,
                                         RayTrav& R, uint32_t* flags) {
    const float BIG = 1e16f;
    f3 inv;
    inv.x = fabs_(dir.x) < 1e-16f ? (dir.x > 0.0f ? BIG : -BIG) : 1.0f / dir.x;
    inv.y = fabs_(dir.y) < 1e-16f ? (dir.y > 0.0f ? BIG : -BIG) : 1.0f / dir.y;
    inv.z = fabs_(dir.z) < 1e-16f ? (dir.z > 0.0f ? BIG : -BIG) : 1.0f / dir.z;
    for (;;) {
        const bool on = R.ref != EMPTY_CHILD;
        const bool leaf = on && (R.ref & LEAF_BIT) != 0u;
        const unsigned long long leaves = __ballot(leaf);
        const int nl = __popcll(leaves), nn = __popcll(__ballot(on && !leaf));
        if (nl + nn <= stop) break;
        if (nl * TRAV_LEAF_VOTE >= nn) {
            if constexpr (WAVE) {
                if (nl <= 8) trav_leaves<8>(S, org, dir, tmin, ts, leaves, R);
                else trav_leaves<4>(S, org, dir, tmin, ts, leaves, R);
            } else if (leaf) {
                trav_leaf(S, org, dir, tmin, ts, R);
            }
        } else {
            if (on && !leaf) trav_node<W>(S, org, inv, ts, R, flags);
        }
    }
}

// The hit of a ray that is done; false: a miss.
__device__ __forceinline__ bool trav_hit(const SceneDev& S, f3 org, f3 dir, const RayTrav& R, HitRec& h) {
    if (R.slot < 0 || !(R.best < 3.40282347e38f)) {
        h.facet = -1;
        h.slot = -1;
        h.t = 3.40282347e38f;
        h.tie = false;
        return false;
    }
    float t;
    tri_test(S.tri, R.slot, org, dir, t, h.u, h.v, h.facet);
    h.t = R.best;
    h.slot = R.slot;
    h.tie = R.tie;
    return true;
}

// Closest hit for a ray (origin, direction as stored in the Ray, MinT = tmin,
// MaxT = FLT_MAX).  Returns false on a miss.  *flags bit 2 is set if the
// stack capacity was exceeded (the host sizes it from the tree depth, so
// this never happens for a well-formed build).
template <int W>
__device__ __forceinline__ bool closest_hit(const SceneDev& S, f3 org, f3 dir, float tmin, const TraceStack& ts,
                                            HitRec& h, uint32_t* flags) {
    RayTrav R;
    trav_begin(R);
    trav_run<W, false>(S, org, dir, tmin, ts, 0, R, flags);
    return trav_hit(S, org, dir, R, h);
}
// The same for a whole wave; on: the lane has a ray.
template <int W>
__device__ __forceinline__ bool closest_hit_wave(const SceneDev& S, bool on, f3 org, f3 dir, float tmin,
                                                 const TraceStack& ts, HitRec& h, uint32_t* flags) {
    RayTrav R;
    trav_begin(R);
    if (!on) R.ref = EMPTY_CHILD;
    trav_run<W, true>(S, org, dir, tmin, ts, 0, R, flags);
    return on && trav_hit(S, org, dir, R, h);
}

// ---- calculateGeometry (SPPM.cpp:36-77) ------------------------------------
struct Geom {
    f3 pos, N;
    float uvx, uvy;
    int kind, opaque, is_sppm;
    f3 albedo, radiance;
    float rough, index, absorb, refl, transl;
};

__device__ inline void calc_geometry(const SceneDev& S, const HitRec& h, Geom& g) {
    const float4* tr = S.tri + 3 * h.slot;
    float4 A = tr[0], B = tr[1], C = tr[2];
    f3 p0 = mk(A.x, A.y, A.z), e1 = mk(B.x, B.y, B.z), e2 = mk(C.x, C.y, C.z);
    const float u = h.u, v = h.v;
    g.pos = (e1 * u + e2 * v) + p0;
    const float* nn = S.facet_nrm + 9 * (size_t)h.facet;
    f3 n0 = mk(nn[0], nn[1], nn[2]), n1 = mk(nn[3], nn[4], nn[5]), n2 = mk(nn[6], nn[7], nn[8]);
    g.N = normalized(((n1 - n0) * u + (n2 - n0) * v) + n0);
    const float2* tv = S.facet_uv + 3 * (size_t)h.facet;
    float2 t0 = tv[0], t1 = tv[1], t2 = tv[2];
    g.uvx = ((t1.x - t0.x) * u + (t2.x - t0.x) * v) + t0.x;
    g.uvy = ((t1.y - t0.y) * u + (t2.y - t0.y) * v) + t0.y;
    const DevAttr& a = S.attrs[S.facet_attr[h.facet]];
    g.kind = a.kind;
    g.opaque = a.opaque;
    g.is_sppm = a.is_sppm;
    g.albedo = mk(a.albedo[0], a.albedo[1], a.albedo[2]);
    g.radiance = mk(a.radiance[0], a.radiance[1], a.radiance[2]);
    g.rough = a.rough;
    g.index = a.index;
    g.absorb = a.absorb;
    g.refl = a.refl;
    g.transl = 0.0f;
    if ((double)a.radiance_norm2 > 1e-6) g.albedo = mk(1.0f, 1.0f, 1.0f);
    if (a.tex_rough >= 0) {
        TexDesc td = S.tex[a.tex_rough];
        float4 c = tex_bilinear(S.texels + td.offset, td.width, td.height, g.uvx, g.uvy);
        g.rough = smin(0.8f, smax(0.05f, 0.5f * c.x));
    }
    if (a.tex_albedo >= 0) {
        TexDesc td = S.tex[a.tex_albedo];
        float4 c = tex_bilinear(S.texels + td.offset, td.width, td.height, g.uvx, g.uvy);
        g.albedo = mk(c.x, c.y, c.z);
        g.radiance = g.radiance * g.albedo;
        g.transl = (float)(1.0 - (double)c.w);
    }
    if (a.tex_bump >= 0) {
        TexDesc td = S.tex[a.tex_bump];
        float4 c = tex_bilinear(S.texels + td.offset, td.width, td.height, g.uvx, g.uvy);
        f3 nm = normalized(mk(2.0f * c.x - 1.0f, 2.0f * c.y - 1.0f, 2.0f * c.z - 1.0f));
        nm = normalized(mk(nm.x, nm.z, nm.y));
        f3 E2 = g.N;
        f3 E1 = fabs_(E2.y) > LO_0P9 ? cross(E2, mk(1, 0, 0)) : cross(E2, mk(0, 1, 0));  // (double)|y| > 0.9
        f3 E3 = normalized(cross(E1, E2));
        // Matrix3 with columns E1,E2,E3; inverse via cofactors (Matrix.h:180-211)
        float m[9] = {E1.x, E2.x, E3.x, E1.y, E2.y, E3.y, E1.z, E2.z, E3.z};
        float C[9];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                int r0 = (i == 0) ? 1 : 0, r1 = (i == 2) ? 1 : 2;
                int c0 = (j == 0) ? 1 : 0, c1 = (j == 2) ? 1 : 2;
                float det2 = m[3 * r0 + c0] * m[3 * r1 + c1] - m[3 * r0 + c1] * m[3 * r1 + c0];
                C[3 * i + j] = det2 * (float)(((i + j) % 2) ? -1 : 1);
            }
        float det = m[0] * C[0] + m[3] * C[3] + m[6] * C[6];
        float ix = 1.0f / det;
        // inverse row i = ix * C[:, i] (adjugate = C^T)
        f3 r0 = mk(ix * C[0], ix * C[3], ix * C[6]);
        f3 r1 = mk(ix * C[1], ix * C[4], ix * C[7]);
        f3 r2 = mk(ix * C[2], ix * C[5], ix * C[8]);
        g.N = normalized(mk(dot(r0, nm), dot(r1, nm), dot(r2, nm)));
    }
}

}  // namespace sppm
