// Vertices whose rings the ring kernels do not take from the child numbering
// (cage vertices other than closed rings of four, faces other than quads with
// consecutive halfedges, boundary edge vertices), from a table built once per
// cage: no list made by another kernel, no ring walked.
//
// What bounds them is the chain of dependent loads, not the work: a level
// has a few thousand such vertices, and one thread per vertex that finds its
// fan through the cage and the level's records takes 16-20 us on every level
// however small.  Here each fan entry has its own lane, whose halfedge and
// edge follow from one table record and two shifts, so a wave waits for two
// loads (header, record) and then for its points; the lanes of a vertex
// exchange them through LDS.  The waves ride in the ring kernel's launch, in
// front of its workgroups, where that latency is hidden.  Against the list
// and a kernel of its own per level: points of an icosphere cage with a
// boundary (727 rare vertices, depth 6) 257 -> 142 us, its refinement with
// four times the faces to depth 7 1754 -> 1599 us, the vertex kernel's 8
// waves per SIMD kept (57 registers).  Cages that do not fit the table
// (build_rare_table) keep the list.
#pragma once

#include "cc_fan.h"
#include "cc_fused.h"

namespace cch {

// What the lanes of one wave exchange: per lane its entry's edge point, face
// point, sharpness, edge and halfedge.
struct RareLds {
    float p[6][64];
    float s[64];
    int32_t e[64], h[64];
};

// One lane's place in the table: entry i of a fan of n halfedges with m edge
// entries (n, or n + 1 on a boundary: the last one is the edge of
// prev(last halfedge)); h and e its halfedge and edge at the level.
struct RareLane {
    int32_t v, h, e;
    int n, m, i, g0;   // g0: lane of entry 0
    bool boundary, live;
    __host__ __device__ __forceinline__ int next(int k) const { return k + 1 < m ? k + 1 : 0; }
};

// The entry of lane `lane` of wave `wave` among the level's rare waves
// (rare_waves).
// Items of the table take 4, 8 or 64 lanes; boundary edge vertices 4.
// Level-d entries are the level-1 ones (born at level k: the level-k ones)
// brought down through children 0: halfedge x becomes 4x, its edge
// 2e + (x > twin(x) ? 0 : 1), and that comparison has the same result on
// every level (see structural_ring).
__host__ __device__ __forceinline__ RareLane rare_lane(const RareView &r, const LevelTab &t, int d, int32_t wave,
                                                       int lane) {
    const int32_t per = (1 << d) - 1;   // boundary edge vertices per boundary halfedge of the cage
    const int32_t q4 = r.n4 + r.nb * per;
    const int32_t w4 = (q4 + 15) >> 4, w8 = (r.n8 + 7) >> 3;
    int lg = 6;
    int32_t it = wave - w4 - w8, base = r.n4 + r.n8, count = r.n64;
    if (wave < w4) {
        lg = 2;
        it = wave * 16 + (lane >> 2);
        base = 0;
        count = q4;
    } else if (wave < w4 + w8) {
        lg = 3;
        it = (wave - w4) * 8 + (lane >> 3);
        base = r.n4;
        count = r.n8;
    }
    RareLane L;
    L.i = lane & ((1 << lg) - 1);
    L.g0 = lane - L.i;
    L.live = it < count;
    L.v = L.h = L.e = 0;
    L.n = L.m = 1;
    L.boundary = false;
    if (!L.live) return L;
    int sh = d - 1;
    bool odd;
    if (lg == 2 && it >= r.n4) {
        // The j-th vertex on boundary halfedge b: j + 1 in binary is 1
        // followed by the path from the cage's halfedge to the boundary
        // halfedge p of level k - 1 whose edge was split (0: child 0 of p,
        // edge 2e; 1: child 3 of next(p), edge 2e + 1).
        const int32_t x = it - r.n4, b = x / per, j = x - b * per;
        const int k = 32 - __builtin_clz((uint32_t)(j + 1));
        const int4 q = r.bnd[b];
        int32_t p = q.x, np = q.y, e = q.z;
        for (int s = k - 2; s >= 0; --s) {
            const int bit = ((j + 1) >> s) & 1;
            p = bit ? 4 * np + 3 : 4 * p;
            np = qnext(p);
            e = 2 * e + bit;
        }
        L.v = t.V[k - 1] + t.F[k - 1] + e;
        L.n = 2;
        L.m = 3;
        L.boundary = true;
        sh = d - k;
        // ring 4 next(p) + 3 (edge 2e + 1, on the boundary), 4p + 1 (edge
        // 2E + p, twin 4 next(p) + 2), then the edge 2e of prev(4p + 1)
        L.h = L.i == 0 ? 4 * np + 3 : 4 * p + 1;
        L.e = L.i == 0 ? 2 * e + 1 : (L.i == 1 ? 2 * t.E[k - 1] + p : 2 * e);
        odd = L.i == 1 ? 4 * p + 1 < 4 * np + 2 : L.i != 0;
    } else {
        const int4 hd = r.item[base + it];
        L.v = hd.x;
        L.n = hd.z;
        L.boundary = hd.w != 0;
        L.m = L.n + (L.boundary ? 1 : 0);
        const int2 en = r.ent[hd.y + (L.i < L.m ? L.i : 0)];
        L.h = en.x;
        L.e = en.y & INT32_MAX;
        odd = en.y < 0;
    }
    L.h <<= 2 * sh;
    L.e = (L.e << sh) + (odd ? (1 << sh) - 1 : 0);
    return L;
}

// the entries of one vertex as its lanes left them in LDS
struct FanFromLds {
    const RareLds &x;
    const RareLane &L;
    __device__ __forceinline__ P3 edge(int k) const { return P3{x.p[0][L.g0 + k], x.p[1][L.g0 + k], x.p[2][L.g0 + k]}; }
    __device__ __forceinline__ FanEntry get(int k) const {
        const int q = L.g0 + k, n1 = L.g0 + L.next(k);
        FanEntry e;
        e.E = edge(k);
        e.PE = edge(L.next(k));
        e.F = P3{x.p[3][q], x.p[4][q], x.p[5][q]};
        e.ts = x.s[q];
        e.ps = x.s[n1];
        e.re = x.e[q];
        e.pe = x.e[n1];
        e.r = x.h[q];
        return e;
    }
    __device__ __forceinline__ int32_t key(int k) const { return x.h[L.g0 + k]; }
};

// Vertex points of the rare vertices of wave `wave`: the rules of
// fan_vertex_point in its order of operations.  Scatter rules: every lane
// sums the ring's sharpness itself, forms its own contribution and puts it
// at its rank, and the first lane adds them in that order; gather rules: the
// first lane runs the rule over the entries.
template <int GATHER, int CREASED>
__device__ __forceinline__ void rare_vertices(const FusedArgs &a, const RareView &r, const LevelTab &t, int d,
                                              int32_t wave, RareLds &x) {
    const int lane = (int)(threadIdx.x & 63u);
    const RareLane L = rare_lane(r, t, d, wave, lane);
    P3 old = zero3(), E = zero3(), F = zero3();
    float s = 0.0f;
    if (L.live) {
        old = a.old[L.v];
        E = a.ep[L.e];
        F = a.fp[L.h >> 2];
        s = CREASED ? lsharp(a.cr, a.C, L.e) : 0.0f;
    }
    x.p[0][lane] = E.x; x.p[1][lane] = E.y; x.p[2][lane] = E.z;
    x.p[3][lane] = F.x; x.p[4][lane] = F.y; x.p[5][lane] = F.z;
    x.s[lane] = s;
    x.e[lane] = L.e;
    x.h[lane] = L.h;
    wave_lds_sync();
    const FanFromLds acc{x, L};
    if (GATHER) {
        if (!L.live || L.i != 0) return;
        Fan f;
        f.kind = 0; f.shift = 0; f.n = L.n; f.boundary = L.boundary;
        f.ri = L.n == 2 && L.boundary && L.v >= t.V[0] + t.F[0] ? 1 : 0;   // boundary edge vertices: 4p + 1
        f.a0 = f.a1 = f.a2 = f.a3 = 0;
        a.vp[L.v] = fan_vertex_point<GATHER, CREASED, 0>(f, acc, old);
        return;
    }
    RingParams rp;
    rp.n = (float)L.n; rp.cc = 0.0f; rp.boundary = L.boundary; rp.s1 = rp.s2 = 0.0f; rp.e1 = rp.e2 = -1; rp.sall = 0.0f;
    if (CREASED) {
        for (int k = L.boundary ? 0 : 1; k <= L.n; ++k) {
            const int q = L.g0 + (k < L.m ? k : 0);
            const float se = x.s[q];
            const int32_t ed = x.e[q];
            rp.cc += sgn(se);
            if (se != 0.0f) {
                if (rp.e1 < 0) { rp.s1 = se; rp.e1 = ed; }
                else if (rp.e2 < 0) { rp.s2 = se; rp.e2 = ed; }
            }
            rp.sall += se;
        }
    }
    const int n1 = L.i < L.n ? L.next(L.i) : 0;
    const P3 con = vertex_scatter_contrib(rp, old, E, acc.edge(n1), F, s, x.s[L.g0 + n1], L.e, CREASED);
    int rank = 0;
    for (int k = 0; k < L.n; ++k) rank += x.h[L.g0 + k] < L.h ? 1 : 0;
    wave_lds_sync();   // every lane has read the edge points
    if (L.live && L.i < L.n) {
        x.p[0][L.g0 + rank] = con.x; x.p[1][L.g0 + rank] = con.y; x.p[2][L.g0 + rank] = con.z;
    }
    wave_lds_sync();
    if (!L.live || L.i != 0) return;
    P3 sum = zero3();
    for (int k = 0; k < L.n; ++k) sum = add(sum, acc.edge(k));
    a.vp[L.v] = sum;
}

}  // namespace cch
