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
