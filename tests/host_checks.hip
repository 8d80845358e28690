// Host-side checks of library internals, compiled for the CPU alone by
// test_host_checks.py.
#include <stdlib.h>

#include "../halfedgecatmullclark_amd/csrc/cc_lists.h"

using namespace cch;

// bit 0: the cage has ring lists, 1: CageRings::simple, 2: RareTable::ok
extern "C" int32_t check_rare_table(const cc_Mesh *m) {
    CageRings r;
    RareTable t;
    build_cage_rings(m, r);
    build_rare_table(m, r, t);
    return (r.ok ? 1 : 0) | (r.simple ? 2 : 0) | (t.ok ? 4 : 0);
}

// the byte offset at3 (at3v: vertices) gives element i of 12- and 24-byte records
struct Six { int32_t w[6]; };
extern "C" uint64_t check_at3(int32_t i, int32_t bytes, int32_t vertices) {
    char *base = reinterpret_cast<char *>(uintptr_t(1) << 40);
    const P3 *p = reinterpret_cast<const P3 *>(base);
    Six *q = reinterpret_cast<Six *>(base);
    const void *r = bytes == 12 ? (const void *)(vertices ? at3v(p, i) : at3(p, i))
                                : (const void *)(vertices ? at3v(q, i) : at3(q, i));
    return (uint64_t)(static_cast<const char *>(r) - base);
}

// allocations until one fails (-1: none does), this library's alone
static std::atomic<int64_t> g_left{-1};
void *operator new(size_t n) {
    if (g_left.load() >= 0 && g_left.fetch_sub(1) == 0) throw std::bad_alloc();
    void *p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

// The lists of `count` times the cage with the left-th allocation failing:
// 1 when they are all there, 0 when memory ran out, 2 when lists are missing
// without a word.
extern "C" int32_t check_lists(const cc_Mesh *m, int32_t count, int64_t left) {
    std::vector<const cc_Mesh *> meshes((size_t)count, m);
    std::vector<CageLists> lists((size_t)count);
    g_left = left;
    const bool ok = build_lists(meshes.data(), lists);
    g_left = -1;
    if (!ok) return 0;
    for (const CageLists &l : lists)
        if (!l.r.ok || !l.rt.ok) return 2;
    return 1;
}

// do the lists agree whether one thread or two build them?
extern "C" int32_t check_threads(const cc_Mesh *m) {
    CageRings a, b;
    build_cage_rings(m, a, false);
    build_cage_rings(m, b, true);
    return a.ok == b.ok && a.simple == b.simple && a.voff == b.voff && a.vring == b.vring && a.vbnd == b.vbnd &&
           a.foff == b.foff && a.fring == b.fring && a.ooff == b.ooff && a.out == b.out && a.odd_v == b.odd_v &&
           a.odd_f == b.odd_f && a.bnd == b.bnd && a.odd_v_entries == b.odd_v_entries &&
           a.odd_f_entries == b.odd_f_entries;
}

// owners of the edges of level d, out[e]; returns DCage::by_pair
extern "C" int32_t check_edge_owners(const cc_Mesh *m, int32_t d, int32_t *out) {
    CageRings r;
    build_cage_rings(m, r);
    DCage c = host_cage_view(m);
    c.by_pair = r.by_pair ? 1 : 0;
    Counts n;
    n.init(m->vertexCount, m->halfedgeCount, m->edgeCount, m->faceCount);
    const LevelTab t = level_tab(n);
    for (int32_t e = 0; e < (int32_t)n.E[d]; ++e) {
        out[e] = edge_rep<true>(c, t, e, d);
        if (!is_edge_rep(c, t, e, d, out[e])) return -1;
    }
    return c.by_pair;
}
