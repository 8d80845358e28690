// Library-internal helpers shared by the host and runtime translation units.
#pragma once

#include <vector>

#include <hip/hip_runtime.h>

#include "../../include/CatmullClarkHIP.h"
#include "cc_common.h"
#include "cc_fused.h"

namespace cch {

// thread-local error channel behind ccs_LastError / ccs_LastErrorString
void set_error(int32_t code, const char *msg);
void clear_error();
int32_t last_error();
// reports a HIP failure on the error channel and stderr; true on error
bool hip_failed(hipError_t e, const char *what);

// makes `dev` current for the scope
struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        if (prev != dev) (void)hipSetDevice(dev);
    }
    ~DeviceGuard() {
        int cur = -1;
        if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
    }
};

// true when every cumulative count the reference evaluates in int32 fits
bool ref_counts_fit_int32(const cc_Mesh *cage, int32_t D, const char **why);

// The cage's vertex and face rings as the device walks them (kWalkCap
// steps at most), in CSR form.  `ok` is false when the lists would exceed
// 4 H + V entries (a cage whose walks do not close): the kernels then walk.
struct CageRings {
    std::vector<int32_t> voff, vring, vbnd, foff, fring, ooff, out;
    std::vector<int32_t> fill;   // scratch
    bool ok = false;
    // every listed halfedge leaves its ring's vertex and lies on its ring's face
    bool own = true;
};

// (into r, whose storage a caller with many cages reuses)
inline void build_cage_rings(const cc_Mesh *m, CageRings &r) {
    r.ok = false;
    r.own = true;
    r.vring.clear();
    r.fring.clear();
    const int32_t V = m->vertexCount, F = m->faceCount, H = m->halfedgeCount;
    const CageHe *he = reinterpret_cast<const CageHe *>(m->halfedges);
    const size_t cap = 4 * (size_t)H + (size_t)V;
    r.voff.assign((size_t)V + 1, 0);
    r.vbnd.assign((size_t)V, 0);
    r.foff.assign((size_t)F + 1, 0);
    r.vring.reserve((size_t)H + 1);   // what a cage whose walks close needs
    r.fring.reserve((size_t)H + 1);
    auto valid = [&](int32_t h) { return h >= 0 && h < H; };
    for (int32_t v = 0; v < V; ++v) {
        r.voff[v] = (int32_t)r.vring.size();
        const int32_t p = m->vertexToHalfedgeIDs[v];
        if (!valid(p)) continue;
        r.vring.push_back(p);
        r.own = r.own && he[p].vert == v;
        int32_t n = 1;
        int32_t g = valid(he[p].prev) ? he[he[p].prev].twin : -1;
        for (; g >= 0 && g != p && n < kWalkCap; ++n) {
            if (!valid(g) || r.vring.size() >= cap) return;
            r.vring.push_back(g);
            r.own = r.own && he[g].vert == v;
            g = valid(he[g].prev) ? he[he[g].prev].twin : -1;
        }
        r.vbnd[v] = g < 0 ? 1 : 0;
    }
    r.voff[V] = (int32_t)r.vring.size();
    for (int32_t f = 0; f < F; ++f) {
        r.foff[f] = (int32_t)r.fring.size();
        const int32_t p = m->faceToHalfedgeIDs[f];
        if (!valid(p)) continue;
        r.fring.push_back(p);
        r.own = r.own && he[p].face == f;
        int32_t n = 1;
        for (int32_t it = he[p].next; it != p && n < kWalkCap; it = he[it].next, ++n) {
            if (!valid(it) || r.fring.size() >= cap) return;
            r.fring.push_back(it);
            r.own = r.own && he[it].face == f;
        }
    }
    r.foff[F] = (int32_t)r.fring.size();
    // halfedges by vertex, ascending (a counting sort)
    r.ooff.assign((size_t)V + 1, 0);
    for (int32_t h = 0; h < H; ++h) {
        const int32_t v = he[h].vert;
        if (v < 0 || v >= V) return;
        ++r.ooff[(size_t)v + 1];
    }
    for (int32_t v = 0; v < V; ++v) r.ooff[(size_t)v + 1] += r.ooff[v];
    r.out.assign((size_t)H, 0);
    r.fill.assign(r.ooff.begin(), r.ooff.end() - 1);
    for (int32_t h = 0; h < H; ++h) r.out[(size_t)r.fill[he[h].vert]++] = h;
    r.ok = true;
}

// The rare-vertex table of a cage (RareView) as one run of int32s: items |
// entries | boundary halfedges, item and boundary records of four ints,
// entries of two.  `simple`: every walk closes, links agree, and every vertex,
// edge and face has all its halfedges in its one ring; a tile pass, which
// finishes a vertex from whichever ring closes inside a tile, takes no other
// cage (of two rings at a vertex, both might write it).  `ok` is false when
// the cage does not fit the table (not simple, or a fan of more than 64
// entries): its rare vertices then go through the rare list.
struct RareTable {
    std::vector<int32_t> item, ent, bnd;
    int32_t n4 = 0, n8 = 0, n64 = 0, nb = 0;
    bool ok = false, simple = false;
    bool empty() const { return n4 + n8 + n64 + nb == 0; }
    struct Item { int32_t v, first, n, boundary; };
    std::vector<Item> items[3];   // scratch
    std::vector<char> seen;
};

inline void build_rare_table(const cc_Mesh *m, const CageRings &r, RareTable &t) {
    t.ok = t.simple = false;
    t.n4 = t.n8 = t.n64 = t.nb = 0;
    for (std::vector<int32_t> *x : {&t.item, &t.ent, &t.bnd}) x->clear();
    for (auto &x : t.items) x.clear();
    const int32_t V = m->vertexCount, F = m->faceCount, H = m->halfedgeCount, E = m->edgeCount;
    if (!r.ok || !r.own || (int64_t)r.vring.size() != H || (int64_t)r.fring.size() != H) return;
    const CageHe *he = reinterpret_cast<const CageHe *>(m->halfedges);
    auto valid = [&](int32_t h) { return h >= 0 && h < H; };
    t.seen.assign((size_t)E, 0);
    int32_t pairs = 0;
    for (int32_t h = 0; h < H; ++h) {
        const CageHe &x = he[h];
        if (!valid(x.next) || !valid(x.prev) || x.prev == h || x.next == h || he[x.next].prev != h ||
            x.twin >= H || x.edge < 0 || x.edge >= E || x.face < 0 || x.face >= F)
            return;
        if (x.twin >= 0 && (he[x.twin].twin != h || he[x.twin].edge != x.edge)) return;
        if (h > x.twin) {   // one pair of halfedges, or one boundary halfedge, per edge
            if (t.seen[x.edge]) return;
            t.seen[x.edge] = 1;
            ++pairs;
            if (x.twin < 0) t.bnd.insert(t.bnd.end(), {h, x.next, x.edge, 0});
        }
    }
    if (pairs != E) return;
    bool fits = true;
    auto add_item = [&](int32_t v, int32_t n, int32_t boundary, size_t first) {
        const int32_t entries = n + boundary;
        const int k = entries <= 4 ? 0 : (entries <= 8 ? 1 : 2);
        t.items[k].push_back({v, (int32_t)(first / 2), n, boundary});
        fits = fits && entries <= 64;
    };
    auto add_ent = [&](int32_t h, int32_t e, bool odd) {
        t.ent.push_back(h);
        t.ent.push_back(odd ? (int32_t)((uint32_t)e | 0x80000000u) : e);
    };
    for (int32_t v = 0; v < V; ++v) {
        const int32_t o = r.voff[v], n = r.voff[v + 1] - o;
        if (n != r.ooff[v + 1] - r.ooff[v]) return;
        if (n == 0) continue;   // no halfedge leaves v
        const bool boundary = r.vbnd[v] != 0;
        // A closed ring of four: marked_ring_fan and structural_ring take it
        // (every entry has a twin w, and next(w) is the entry before it).
        if (n == 4 && !boundary) continue;
        const size_t first = t.ent.size();
        for (int32_t i = 0; i < n; ++i) {   // the ring's previous edge is the next entry's edge
            const int32_t R = r.vring[o + i], w = he[R].twin;
            const int32_t tw = w >= 0 ? 4 * he[w].next + 3 : -1;
            add_ent(4 * R, 2 * he[R].edge + (R > w ? 0 : 1), 4 * R < tw);
        }
        if (boundary) {
            const int32_t R = r.vring[o + n - 1], p = he[R].prev;
            add_ent(4 * R, 2 * he[p].edge + 1, true);
        }
        add_item(v, n, boundary ? 1 : 0, first);
    }
    for (int32_t f = 0; f < F; ++f) {
        const int32_t o = r.foff[f], n = r.foff[f + 1] - o;
        if (n == 0) continue;
        const int32_t p = r.fring[o];
        if (p + 3 < H && he[p].next == p + 1 && he[p + 1].next == p + 2 && he[p + 2].next == p + 3 &&
            he[p + 3].next == p)
            continue;
        const size_t first = t.ent.size();
        for (int32_t i = 0; i < n; ++i) {
            const int32_t q = r.fring[o + i], pr = he[q].prev;
            add_ent(4 * q + 2, 2 * E + pr, 4 * q + 2 < 4 * pr + 1);
        }
        add_item(V + f, n, 0, first);
    }
    t.simple = true;
    if (!fits) return;
    for (const auto &group : t.items) {
        const int32_t *p = reinterpret_cast<const int32_t *>(group.data());
        t.item.insert(t.item.end(), p, p + 4 * group.size());
    }
    t.n4 = (int32_t)t.items[0].size();
    t.n8 = (int32_t)t.items[1].size();
    t.n64 = (int32_t)t.items[2].size();
    t.nb = (int32_t)(t.bnd.size() / 4);
    t.ok = true;
}

// host-memory view of a cage with the device-view type (for the O(depth) maps)
inline DCage host_cage_view(const cc_Mesh *m) {
    DCage c;
    c.vring_off = c.vring = c.vring_bnd = c.fring_off = c.fring = c.vout_off = c.vout = nullptr;
    c.he = reinterpret_cast<const CageHe *>(m->halfedges);
    c.v2h = m->vertexToHalfedgeIDs;
    c.e2h = m->edgeToHalfedgeIDs;
    c.f2h = m->faceToHalfedgeIDs;
    c.pts = reinterpret_cast<const P3 *>(m->vertexPoints);
    c.uvs = reinterpret_cast<const UV *>(m->uvs);
    c.cr = reinterpret_cast<const Crease *>(m->creases);
    c.V = m->vertexCount; c.U = m->uvCount; c.H = m->halfedgeCount; c.E = m->edgeCount; c.F = m->faceCount;
    return c;
}

inline LevelTab level_tab(const Counts &n) {
    LevelTab t;
    for (int d = 0; d <= kMaxDepth; ++d) {
        t.E[d] = (int32_t)n.E[d];
        t.V[d] = (int32_t)n.V[d];
        t.F[d] = (int32_t)n.F[d];
    }
    int64_t words = 0;   // levels past the addressable range are never used
    t.R[0] = 0;
    for (int d = 1; d <= kMaxDepth; ++d) {
        t.R[d] = (int32_t)std::min<int64_t>(words, INT32_MAX);
        words += (n.H[d] + 63) / 64;
    }
    return t;
}

}  // namespace cch
