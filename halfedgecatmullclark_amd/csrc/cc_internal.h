// Library-internal helpers shared by the host and runtime translation units.
#pragma once

#include <atomic>
#include <exception>
#include <new>
#include <thread>
#include <utility>
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
// The walks also say whether the cage is `simple`: every walk closes, links
// agree, and every vertex, edge and face has all its halfedges in its one
// ring.  A tile pass, which finishes a vertex from whichever ring closes
// inside a tile, takes no other cage (of two rings at a vertex, both might
// write it).  The tests read nothing that a walk does not read anyway (a pass
// of their own over 524 thousand halfedges took half as long as the walks).
struct CageRings {
    std::vector<int32_t> voff, vring, vbnd, foff, fring, ooff, out;
    // vertices other than closed rings of four, faces other than quads with
    // consecutive halfedges, boundary halfedges
    std::vector<int32_t> odd_v, odd_f, bnd;
    std::vector<int32_t> fill;   // scratch
    std::vector<uint8_t> seen;
    bool ok = false, simple = false;
    bool by_pair = true;   // DCage::by_pair
    bool pairs[2] = {};    // as the vertices' and the edges' part find it
    int64_t odd_v_entries = 0, odd_f_entries = 0;   // entries the rare-vertex table would have
    bool part_ok[3] = {};
    // of each part, any bit: not simple (gathered without branches)
    int32_t bad[3] = {};
};

inline void ring_vertices(const cc_Mesh *m, CageRings &r) {
    const int32_t V = m->vertexCount, H = m->halfedgeCount;
    // (in variables of this thread's own: the lists' headers share cache lines)
    std::vector<int32_t> voff = std::move(r.voff), vring = std::move(r.vring), vbnd = std::move(r.vbnd), odd_v = std::move(r.odd_v);
    const CageHe *he = reinterpret_cast<const CageHe *>(m->halfedges);
    const size_t cap = 4 * (size_t)H + (size_t)V;
    auto valid = [&](int32_t h) { return h >= 0 && h < H; };
    int32_t bad = 0;
    int64_t entries = 0;
    bool by_pair = false;
    voff.assign((size_t)V + 1, 0);
    vbnd.assign((size_t)V, 0);
    vring.clear();
    odd_v.clear();
    vring.reserve((size_t)H + 1);   // what a cage whose walks close needs
    // twin(prev(h)), -1 without; a ring's step agrees when that twin's twin is
    // prev(h) again and both have one edge
    auto step = [&](int32_t h) {
        const int32_t q = he[h].prev;
        if (!valid(q)) {
            bad = 1;
            return -1;
        }
        const int32_t g = he[q].twin;
        if (valid(g)) {
            bad |= (he[g].twin ^ q) | (he[g].edge ^ he[q].edge);
            by_pair |= q > g && (q <= he[g].next || h < g);   // (h is next(q))
        }
        return g;
    };
    for (int32_t v = 0; v < V; ++v) {
        voff[v] = (int32_t)vring.size();
        const int32_t p = m->vertexToHalfedgeIDs[v];
        if (!valid(p)) continue;
        vring.push_back(p);
        bad |= he[p].vert ^ v;
        int32_t n = 1;
        int32_t g = step(p);
        for (; g >= 0 && g != p && n < kWalkCap; ++n) {
            if (!valid(g) || vring.size() >= cap) return;
            vring.push_back(g);
            bad |= he[g].vert ^ v;
            g = step(g);
        }
        vbnd[v] = g < 0 ? 1 : 0;
        if (n != 4 || g < 0) {
            odd_v.push_back(v);
            entries += n + (g < 0 ? 1 : 0);
        }
    }
    voff[V] = (int32_t)vring.size();
    r.odd_v_entries = entries;
    r.pairs[0] = by_pair;
    r.bad[0] = bad | ((int64_t)vring.size() != H ? 1 : 0);
    r.voff = std::move(voff);
    r.vring = std::move(vring);
    r.vbnd = std::move(vbnd);
    r.odd_v = std::move(odd_v);
    r.part_ok[0] = true;
}

inline void ring_faces(const cc_Mesh *m, CageRings &r) {
    const int32_t V = m->vertexCount, F = m->faceCount, H = m->halfedgeCount;
    std::vector<int32_t> foff = std::move(r.foff), fring = std::move(r.fring), odd_f = std::move(r.odd_f);
    const CageHe *he = reinterpret_cast<const CageHe *>(m->halfedges);
    const size_t cap = 4 * (size_t)H + (size_t)V;
    auto valid = [&](int32_t h) { return h >= 0 && h < H; };
    int32_t bad = 0;
    int64_t entries = 0;
    foff.assign((size_t)F + 1, 0);
    fring.clear();
    odd_f.clear();
    fring.reserve((size_t)H + 1);
    for (int32_t f = 0; f < F; ++f) {
        foff[f] = (int32_t)fring.size();
        const int32_t p = m->faceToHalfedgeIDs[f];
        if (!valid(p)) continue;
        fring.push_back(p);
        bad |= he[p].face ^ f;
        int32_t n = 1, last = p;
        for (int32_t it = he[p].next; it != p && n < kWalkCap; it = he[it].next, ++n) {
            if (!valid(it) || fring.size() >= cap) return;
            fring.push_back(it);
            bad |= (he[it].face ^ f) | (he[it].prev ^ last);
            last = it;
        }
        bad |= (he[p].prev ^ last) | (n < 2 ? 1 : 0);
        if (n != 4 || he[p].next != p + 1 || he[p + 1].next != p + 2 || he[p + 2].next != p + 3) {
            odd_f.push_back(f);
            entries += n;
        }
    }
    foff[F] = (int32_t)fring.size();
    r.odd_f_entries = entries;
    r.bad[1] = bad | ((int64_t)fring.size() != H ? 1 : 0);
    r.foff = std::move(foff);
    r.fring = std::move(fring);
    r.odd_f = std::move(odd_f);
    r.part_ok[1] = true;
}

// halfedges by vertex, ascending (a counting sort); an edge has one pair of
// halfedges or one boundary halfedge
inline void ring_out(const cc_Mesh *m, CageRings &r) {
    const int32_t V = m->vertexCount, H = m->halfedgeCount, E = m->edgeCount;
    std::vector<int32_t> ooff = std::move(r.ooff), out = std::move(r.out), fill = std::move(r.fill), bnd = std::move(r.bnd);
    std::vector<uint8_t> seen = std::move(r.seen);
    const CageHe *he = reinterpret_cast<const CageHe *>(m->halfedges);
    ooff.assign((size_t)V + 1, 0);
    seen.assign((size_t)(E > 0 ? E : 0), 0);
    bnd.clear();
    int32_t bad = 0, pairs = 0;
    bool by_pair = false;
    for (int32_t h = 0; h < H; ++h) {
        const CageHe &x = he[h];
        if (x.vert < 0 || x.vert >= V) return;
        ++ooff[(size_t)x.vert + 1];
        if (x.edge < 0 || x.edge >= E) {
            bad = 1;
        } else {
            seen[x.edge] += h > x.twin ? 1 : 0;
            by_pair |= h > x.twin && m->edgeToHalfedgeIDs[x.edge] != h;
        }
        pairs += h > x.twin ? 1 : 0;
        if (x.twin < 0) bnd.push_back(h);
    }
    for (const uint8_t n : seen) bad |= n ^ 1;   // (modulo 256; with E pairs in all, one each)
    for (int32_t v = 0; v < V; ++v) ooff[(size_t)v + 1] += ooff[v];
    out.assign((size_t)H, 0);
    fill.assign(ooff.begin(), ooff.end() - 1);
    for (int32_t h = 0; h < H; ++h) out[(size_t)fill[he[h].vert]++] = h;
    r.pairs[1] = by_pair;
    r.bad[2] = bad | (pairs ^ E);
    r.ooff = std::move(ooff);
    r.out = std::move(out);
    r.fill = std::move(fill);
    r.bnd = std::move(bnd);
    r.seen = std::move(seen);
    r.part_ok[2] = true;
}

// (into r, whose storage a caller with many cages reuses)
// threads: a second one for the faces and the outgoing halfedges of a cage of
// at least kRingThreadsFrom halfedges (the lists of 524 thousand halfedges 3.33
// ms on one and 1.85 on two, of 45 thousand 0.44 and 0.28; at 16 thousand a
// whole host call to depth 1 took 0.27 ms with one and 0.30 with two)
constexpr int32_t kRingThreadsFrom = 1 << 15;
inline void build_cage_rings(const cc_Mesh *m, CageRings &r, bool threads = false) {
    for (bool &x : r.part_ok) x = false;
    r.ok = r.simple = false;
    r.by_pair = true;
    std::atomic<bool> memory{true};
    auto rest = [&]() {   // no exception leaves a thread
        try {
            ring_faces(m, r);
            ring_out(m, r);
        } catch (const std::bad_alloc &) {
            memory = false;
        }
    };
    std::thread other;
    if (threads && m->halfedgeCount >= kRingThreadsFrom) {
        try {
            other = std::thread(rest);
        } catch (const std::exception &) {   // no thread to be had: done below
        }
    }
    try {
        ring_vertices(m, r);
    } catch (const std::bad_alloc &) {
        memory = false;
    }
    if (other.joinable()) other.join();
    else rest();
    if (!memory) throw std::bad_alloc();
    r.ok = r.part_ok[0] && r.part_ok[1] && r.part_ok[2];
    if (!r.ok) return;
    // (rings of as many halfedges as the cage has, none of them twice: all)
    int32_t bad = r.bad[0] | r.bad[1] | r.bad[2];
    for (int32_t v = 0; v < m->vertexCount; ++v)   // all of v's in its ring
        bad |= (r.voff[v + 1] - r.voff[v]) ^ (r.ooff[v + 1] - r.ooff[v]);
    r.simple = bad == 0;
    r.by_pair = !r.simple || r.pairs[0] || r.pairs[1];
}

// The rare-vertex table of a cage (RareView) as one run of int32s: items |
// entries | boundary halfedges, item and boundary records of four ints,
// entries of two.  `ok` is false when the cage does not fit it (not simple, or
// a fan of more than 64 entries): its rare vertices then go through the rare
// list.
struct RareTable {
    std::vector<int32_t> item, ent, bnd;
    int32_t n4 = 0, n8 = 0, n64 = 0, nb = 0;
    bool ok = false;
    bool empty() const { return n4 + n8 + n64 + nb == 0; }
    void clear() {
        ok = false;
        n4 = n8 = n64 = nb = 0;
        for (std::vector<int32_t> *x : {&item, &ent, &bnd}) x->clear();
        for (auto &x : items) x.clear();
    }
    struct Item { int32_t v, first, n, boundary; };
    std::vector<Item> items[3];   // scratch
};

inline void build_rare_table(const cc_Mesh *m, const CageRings &r, RareTable &t) {
    t.clear();
    if (!r.ok || !r.simple) return;
    const int32_t V = m->vertexCount, E = m->edgeCount;
    const CageHe *he = reinterpret_cast<const CageHe *>(m->halfedges);
    bool fits = true;
    auto add_item = [&](int32_t v, int32_t n, int32_t boundary, size_t first) {
        const int32_t entries = n + boundary;
        const int k = entries <= 4 ? 0 : (entries <= 8 ? 1 : 2);
        t.items[k].push_back({v, (int32_t)(first / 2), n, boundary});
        fits = fits && entries <= 64;
    };
    std::vector<int32_t> ent = std::move(t.ent);
    ent.reserve(2 * (size_t)(r.odd_v_entries + r.odd_f_entries));
    auto add_ent = [&](int32_t h, int32_t e, bool odd) {
        ent.push_back(h);
        ent.push_back(odd ? (int32_t)((uint32_t)e | 0x80000000u) : e);
    };
    // (a closed ring of four marked_ring_fan and structural_ring take: every
    // entry R has a twin w, and next(w) is the entry before it)
    for (const int32_t v : r.odd_v) {
        const int32_t o = r.voff[v], n = r.voff[v + 1] - o;
        const bool boundary = r.vbnd[v] != 0;
        const size_t first = ent.size();
        int32_t before = boundary ? -1 : r.vring[o + n - 1];
        for (int32_t i = 0; i < n; ++i) {   // the ring's previous edge is the next entry's edge
            const int32_t R = r.vring[o + i];
            const CageHe &x = he[R];
            add_ent(4 * R, 2 * x.edge + (R > x.twin ? 0 : 1), R <= before);   // child 0's twin is 4 before + 3
            before = R;
        }
        if (boundary) add_ent(4 * before, 2 * he[he[before].prev].edge + 1, true);
        add_item(v, n, boundary ? 1 : 0, first);
        if (!fits) return;
    }
    for (const int32_t f : r.odd_f) {
        const int32_t o = r.foff[f], n = r.foff[f + 1] - o;
        const size_t first = ent.size();
        int32_t pr = r.fring[o + n - 1];
        for (int32_t i = 0; i < n; ++i) {
            const int32_t q = r.fring[o + i];
            add_ent(4 * q + 2, 2 * E + pr, q < pr);   // 4 q + 2 < 4 pr + 1
            pr = q;
        }
        add_item(V + f, n, 0, first);
        if (!fits) return;
    }
    t.ent = std::move(ent);
    for (const int32_t h : r.bnd) t.bnd.insert(t.bnd.end(), {h, he[h].next, he[h].edge, 0});
    for (const auto &group : t.items) {
        const int32_t *p = reinterpret_cast<const int32_t *>(group.data());
        t.item.insert(t.item.end(), p, p + 4 * group.size());
    }
    t.n4 = (int32_t)t.items[0].size();
    t.n8 = (int32_t)t.items[1].size();
    t.n64 = (int32_t)t.items[2].size();
    t.nb = (int32_t)r.bnd.size();
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
