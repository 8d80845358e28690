// Host-side checks of library internals, compiled for the CPU alone by
// test_host_checks.py.
#include "../halfedgecatmullclark_amd/csrc/cc_internal.h"

using namespace cch;

// bit 0: the cage has ring lists, 1: RareTable::simple, 2: RareTable::ok
extern "C" int32_t check_rare_table(const cc_Mesh *m) {
    CageRings r;
    RareTable t;
    build_cage_rings(m, r);
    build_rare_table(m, r, t);
    return (r.ok ? 1 : 0) | (t.simple ? 2 : 0) | (t.ok ? 4 : 0);
}

// the byte offset at3 gives element i of 12- and 24-byte records
struct Six { int32_t w[6]; };
extern "C" uint64_t check_at3(int32_t i, int32_t bytes) {
    char *base = reinterpret_cast<char *>(uintptr_t(1) << 40);
    const void *p = bytes == 12 ? (const void *)at3(reinterpret_cast<const P3 *>(base), i)
                                : (const void *)at3(reinterpret_cast<Six *>(base), i);
    return (uint64_t)(static_cast<const char *>(p) - base);
}
