// Points of one level (d >= 2) tile by tile, topology untouched: face points
// (CatmullClark.h:2004-2052), edge points (:2065-2241) and, for the vertices
// whose ring of four closes inside the tile, vertex points (:2254-2615).
//
// One thread takes one quad: the children 4p .. 4p+3 of a level-(d-1)
// halfedge p.  Its records follow from p's without a select, two of its four
// edges and its face vertex are shared with the other lanes of p's own quad
// (DPP), and only the two halves of p's edge and of prev(p)'s go through LDS.
// A tile of N quads is a square patch (16 x 16 or 32 x 32), and most of its
// vertices have their whole ring inside it; a vertex kernel of its own reads
// every face and edge point back for them (1.6 GB at level 7 of the 64 x 32
// torus).  The representatives of the others, and of vertices with a creased
// edge, are left to the masked vertex kernel ("far" bits) and the rare-vertex
// table.  Every sum runs in the order of the other kernels (edge points add
// two terms, which commute), so the points are the same bit for bit.
//
// What bounds it: with a halfedge or two per lane the instructions (457 per
// lane and two halfedges, three quarters of the issue slots), with a quad per
// lane (about 400 for four) the 2.55 GB it moves, as long as nothing spills
// (20 spilled registers: 1450 us).  Level 7 of the torus, tile kernel and far
// vertices: 1059 + 642 us with the fused kernel and every vertex read back,
// 1036 + 372 one halfedge at a time, 612 + 345 with tiles of 512 quads, 596 +
// 277 with 1024 (half as many vertices lie on an edge); over runs and boxes
// 596-650 + 276-282.  Only cages whose vertices have one ring each come here
// (CageRings::simple): whichever ring closes in a tile writes its vertex.
#pragma once

#include "cc_level.h"

namespace cch {

// a point of an LDS array of N points, by component: a lane's address is one
// shift (twelve-byte records take a quarter-rate multiplication each)
template <int N>
__device__ __forceinline__ P3 tile_get(const float (&s)[3][N], int i) {
    return P3{s[0][i], s[1][i], s[2][i]};
}
template <int N>
__device__ __forceinline__ void tile_put(float (&s)[3][N], int i, P3 p) {
    s[0][i] = p.x;
    s[1][i] = p.y;
    s[2][i] = p.z;
}
template <int CTRL>
__device__ __forceinline__ P3 quad_rel3(P3 p) {
    return P3{quad_relf<CTRL>(p.x), quad_relf<CTRL>(p.y), quad_relf<CTRL>(p.z)};
}

// the gather rules' point of a smooth vertex with the ring's face points F
// and own edges' points E in fan order
template <int CREASED>
__device__ __forceinline__ P3 smooth_gather4(const P3 (&F)[4], const P3 (&E)[4], P3 old) {
    FanEntry en[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        en[k].r = k;
        en[k].re = en[k].pe = 0;
        en[k].E = E[k];
        en[k].PE = E[(k + 1) & 3];
        en[k].F = F[k];
        en[k].ts = en[k].ps = 0.0f;
    }
    Fan f;
    f.kind = 1; f.shift = 0; f.n = 4; f.ri = 0; f.boundary = false;
    f.a0 = f.a1 = f.a2 = f.a3 = 0;
    return fan_vertex_point<1, CREASED, 4>(f, FanPreloaded{en[0], en[1], en[2], en[3]}, old);
}

template <int GATHER, int CREASED, int N>
__device__ __forceinline__ void point_tile(const FusedArgs &a, uint32_t tile) {
    __shared__ float sA[3][N];                // scatter: child 0's side of its edge; gather: the face point
    __shared__ float sB[3][GATHER ? 1 : N];   // scatter: child 3's side
    __shared__ float sC[3][N];                // scatter: child 0's share of its vertex; gather: its edge point
    __shared__ float sD[3][N];                // scatter: the pair sum of p's edge vertex; gather: child 1's edge point
    __shared__ int32_t sring[N];              // twin(prev(p)), the next of p's ring; -1 across a creased edge
    __shared__ uint16_t flist[2 * N];         // outer edges written into another tile: 2 quad + (child 3)
    __shared__ int32_t nfar;
    const int q = (int)threadIdx.x;
    if (q == 0) nfar = 0;
    // the masked kernel that follows appends; on this path no fused kernel
    // with points has emptied the list of the level before
    if (a.rare && tile == 0 && q == 0) a.rare[0] = 0;
    const int32_t base = (int32_t)(tile * N), p = base + q;
    const auto here = [&](int32_t r) { return (uint32_t)(r - base) < (uint32_t)N; };
    const auto sharp = [&](int32_t e) {
        const bool has = e < a.C;   // a level's crease array is never empty
        const float cs = gld(&at3(a.cr, has ? e : 0)->sharp);
        return has ? cs : 0.0f;
    };
    const bool live = p < a.F;           // a multiple of 4: parent quads are whole
    const int32_t g = live ? p : p & 3;
    const int4 r = he_gld(a.par, g);
    __syncthreads();   // nfar
    const int32_t w = r.x, wp = quad_rel<kQuadPrev>(w), gp = qprev(g);
    const int32_t e0 = 2 * r.y + (g > w ? 0 : 1), e3 = 2 * quad_rel<kQuadPrev>(r.y) + (gp > wp ? 1 : 0);
    const int32_t v1 = a.pV + a.pF + r.y, v2 = a.pV + (g >> 2);
    const P3 P0 = gld(at3v(a.old, r.z)), P1 = gld(at3v(a.old, v1)), P2 = gld(at3v(a.old, v2));
    float s0 = 0.0f, s3 = 0.0f;          // (edges inside p's quad have no sharpness)
    if (CREASED && __any(e0 < a.C || e3 < a.C)) {
        s0 = sharp(e0);
        s3 = sharp(e3);
    }
    const bool in0 = w >= 0 && here(w), in3 = wp >= 0 && here(wp);
    const bool own0 = live && g > qnext(w), own3 = live && g >= wp;   // the larger of the pair writes the edge
    if (w >= 0 && !in0 && own0) flist[atomicAdd(&nfar, 1)] = (uint16_t)(2 * q);
    if (wp >= 0 && !in3 && own3) flist[atomicAdd(&nfar, 1)] = (uint16_t)(2 * q + 1);
    const P3 P3_ = quad_rel3<kQuadPrev>(P1);
    const P3 F = face_rule(P0, P1, P2, P3_, GATHER);
    if (live) *at3(a.fp, p) = F;
    P3 E1;
    if (GATHER) {
        tile_put(sA, q, F);
        E1 = edge_gather(P1, P2, F, quad_rel3<kQuadNext>(F), CREASED ? 0.0f : 1.0f, CREASED);
    } else {
        tile_put(sA, q, edge_contrib(P0, P1, F, false, s0, CREASED));
        tile_put(sB, q, edge_contrib(P3_, P0, F, false, s3, CREASED));
        const P3 m1 = edge_contrib(P1, P2, F, false, 0.0f, CREASED);
        const P3 m2 = edge_contrib(P2, P3_, F, false, 0.0f, CREASED);
        E1 = add(add(zero3(), m1), quad_rel3<kQuadNext>(m2));
    }
    if (live) *at3(a.ep + 2 * (int64_t)a.pE, p) = E1;
    __syncthreads();
    P3 E0, E3;
    {
        const P3 o0 = in0 ? (GATHER ? tile_get(sA, qnext(w) - base) : tile_get(sB, qnext(w) - base)) : zero3();
        const P3 o3 = in3 ? tile_get(sA, wp - base) : zero3();
        if (GATHER) {
            E0 = edge_gather(P0, P1, F, o0, CREASED ? sat(s0) : 1.0f, CREASED);
            E3 = edge_gather(P3_, P0, F, o3, CREASED ? sat(s3) : 1.0f, CREASED);
        } else {
            E0 = add(add(zero3(), o0), tile_get(sA, q));
            E3 = add(add(zero3(), o3), tile_get(sB, q));
        }
    }
    if (__any(w < 0 || wp < 0)) {
        const P3 P3_ = quad_rel3<kQuadPrev>(P1);
        if (GATHER) {   // (the reference's second face point is that of face 0)
            const P3 Z = quad_face(a.he, a.old, 0, true);
            if (w < 0) E0 = edge_gather(P0, P1, F, Z, CREASED ? sat(s0) : 0.0f, CREASED);
            if (wp < 0) E3 = edge_gather(P3_, P0, F, Z, CREASED ? sat(s3) : 0.0f, CREASED);
        } else {
            if (w < 0) E0 = add(zero3(), edge_contrib(P0, P1, F, true, s0, CREASED));
            if (wp < 0) E3 = add(zero3(), edge_contrib(P3_, P0, F, true, s3, CREASED));
        }
    }
    if (live && (w < 0 || (in0 && own0))) *at3(a.ep, e0) = E0;
    if (live && (wp < 0 || (in3 && own3))) *at3(a.ep, e3) = E3;

    // p's edge vertex is finished here when twin(p) is in the tile (in
    // another quad) and both halves of the edge are smooth
    const bool smooth = s0 == 0.0f && quad_relf<kQuadNext>(s3) == 0.0f;
    const bool done1 = in0 && smooth && (g >> 2) != (w >> 2);
    sring[q] = live && s3 == 0.0f ? wp : -1;
    P3 c0 = zero3(), a1 = zero3(), a2 = zero3();
    if (GATHER) {
        tile_put(sC, q, E0);
        tile_put(sD, q, E1);
    } else {
        RingParams rp;   // of a smooth vertex with four edges
        rp.n = 4.0f; rp.cc = 0.0f; rp.boundary = false; rp.s1 = rp.s2 = 0.0f; rp.e1 = rp.e2 = -1; rp.sall = 0.0f;
        const auto share = [&](P3 P, P3 E, P3 Fq) {
            return vertex_scatter_contrib(rp, P, E, zero3(), Fq, 0.0f, 0.0f, 0, CREASED);
        };
        c0 = share(P0, E0, F);
        tile_put(sC, q, c0);
        // p's edge vertex: child 1 of p and child 3 of next(p), ascending
        const P3 c1 = share(P1, E1, F), c3 = share(P1, quad_rel3<kQuadNext>(E3), quad_rel3<kQuadNext>(F));
        const bool wrap = (g & 3) == 3;
        a1 = wrap ? c3 : c1;
        a2 = wrap ? c1 : c3;
        tile_put(sD, q, add(add(zero3(), a1), a2));
        // the face vertex of p's quad: its four children 2, ascending
        const P3 E2 = quad_rel3<kQuadPrev>(E1);
        const P3 c2 = share(P2, E2, F);
        const P3 v = add(add(add(add(zero3(), quad_bcast3<0>(c2)), quad_bcast3<1>(c2)), quad_bcast3<2>(c2)),
                         quad_bcast3<3>(c2));
        if (live && (g & 3) == 0) *at3v(a.vp, v2) = v;
    }
    if (GATHER) {
        const P3 E2 = quad_rel3<kQuadPrev>(E1);
        const P3 Fq[4] = {quad_bcast3<0>(F), quad_bcast3<1>(F), quad_bcast3<2>(F), quad_bcast3<3>(F)};
        const P3 Eq[4] = {quad_bcast3<0>(E2), quad_bcast3<1>(E2), quad_bcast3<2>(E2), quad_bcast3<3>(E2)};
        const P3 v = smooth_gather4<CREASED>(Fq, Eq, P2);
        if (live && (g & 3) == 0) *at3v(a.vp, v2) = v;
    }
    // the level's owner bits, four of each lane
    uint32_t own = 0;
    if (live) own = (uint32_t)(a.own_in[p >> 4] >> (4 * (p & 15))) & 15u;
    __syncthreads();

    // p's edge vertex: the gather rules start from its representative, the
    // scatter rules add the smaller quad's pair and then the larger's two
    if (GATHER) {
        const P3 Fn = quad_rel3<kQuadNext>(F), E3n = quad_rel3<kQuadNext>(E3);
        if (done1 && (own & 2u) != 0u) {
            const P3 Fq[4] = {F, tile_get(sA, qnext(w) - base), tile_get(sA, w - base), Fn};
            const P3 Eq[4] = {E1, E0, tile_get(sD, w - base), E3n};
            *at3v(a.vp, v1) = smooth_gather4<CREASED>(Fq, Eq, P1);
        }
    } else if (live && done1 && g > w) {
        *at3v(a.vp, v1) = add(add(tile_get(sD, w - base), a1), a2);
    }
    // p's vertex: p's ring, four times x -> twin(prev(x))
    const int32_t r1 = sring[q];
    bool ring = live && here(r1);
    const int32_t r2 = ring ? sring[r1 - base] : -1;
    ring = ring && here(r2);
    const int32_t r3 = ring ? sring[r2 - base] : -1;
    ring = ring && here(r3);
    const int32_t r4 = ring ? sring[r3 - base] : -1;
    ring = ring && r4 == g && r2 != g;   // four distinct halfedges
    {   // the representatives left over, 16 lanes a word
        const uint32_t nib = own & ~((ring ? 1u : 0u) | (done1 ? 2u : 0u) | 4u);
        const uint32_t sh = 4u * (uint32_t)(q & 7);
        const uint32_t lo = row_or((q & 8) ? 0u : nib << sh);
        const uint32_t hi = row_or((q & 8) ? nib << sh : 0u);
        if ((q & 15) == 15 && (p & ~15) < a.F) a.far[p >> 4] = ((uint64_t)hi << 32) | lo;
    }
    if (GATHER) {
        if (ring && (own & 1u) != 0u) {
            const int32_t x1 = r1 - base, x2 = r2 - base, x3 = r3 - base;
            const P3 Fq[4] = {F, tile_get(sA, x1), tile_get(sA, x2), tile_get(sA, x3)};
            const P3 Eq[4] = {E0, tile_get(sC, x1), tile_get(sC, x2), tile_get(sC, x3)};
            *at3v(a.vp, r.z) = smooth_gather4<CREASED>(Fq, Eq, P0);
        }
    } else if (ring && g < r1 && g < r2 && g < r3) {   // shares in ascending halfedge order
        const int32_t lo = r1 < r2 ? r1 : r2, hi = r1 < r2 ? r2 : r1;
        const int32_t x3 = hi > r3 ? hi : r3, m = hi > r3 ? r3 : hi;
        const int32_t x1 = lo < m ? lo : m, x2 = lo < m ? m : lo;
        *at3v(a.vp, r.z) = add(add(add(add(zero3(), c0), tile_get(sC, x1 - base)), tile_get(sC, x2 - base)),
                              tile_get(sC, x3 - base));
    }
    // Outer edges whose twin lies in another tile, one lane each (every wave
    // going through this for its own few would be a third of the kernel's
    // instructions; last, when nothing else is held in registers): the twin's side from the corners of its quad t, two of
    // which are the edge's ends.
    const int32_t n = nfar;
    for (int32_t i = (int32_t)((threadIdx.x + 64 * tile) & (N - 1)); i < n; i += N) {
        const int32_t k = flist[i], f = base + (k >> 1);
        const bool last = (k & 1) != 0;
        const int4 y = he_gld(a.par, last ? qprev(f) : f);
        const int32_t t = last ? y.x : qnext(y.x);
        const int32_t e = 2 * y.y + ((last ? qprev(f) : f) > y.x ? 0 : 1);
        const int4 y0 = he_gld(a.par, t), y3 = he_gld(a.par, qprev(t));
        const P3 Q0 = gld(at3v(a.old, y0.z)), Q1 = gld(at3v(a.old, a.pV + a.pF + y0.y));
        const P3 Q2 = gld(at3v(a.old, a.pV + (t >> 2))), Q3 = gld(at3v(a.old, a.pV + a.pF + y3.y));
        const int32_t ee = last ? (e ^ 1) : e;
        const float ts = CREASED ? sharp(ee) : 0.0f;
        const P3 Ft = face_rule(Q0, Q1, Q2, Q3, GATHER);
        // child 0 of f meets child 3 of t (from Q3 to Q0), child 3 of f child 0 of t
        const P3 t0 = last ? Q0 : Q3, t1 = last ? Q1 : Q0;
        P3 E;
        if (GATHER)
            E = edge_gather(t1, t0, tile_get(sA, k >> 1), Ft, CREASED ? sat(ts) : 1.0f, CREASED);
        else
            E = add(add(zero3(), edge_contrib(t0, t1, Ft, false, ts, CREASED)),
                    last ? tile_get(sB, k >> 1) : tile_get(sA, k >> 1));
        *at3(a.ep, ee) = E;
    }
}

}  // namespace cch
