// The host lists of many cages at once (ccb_Create).
#pragma once

#include <algorithm>
#include <atomic>
#include <exception>
#include <new>
#include <thread>
#include <vector>

#include "cc_internal.h"

namespace cch {

struct CageLists {
    CageRings r;
    RareTable rt;
};

// Every cage's ring lists and rare-vertex table.  The walks wait for one
// cached halfedge after another (48 cages of 535 thousand halfedges: 22 ms on
// one core), and the cages are independent: up to eight threads take them in
// turn, one per 16 thousand halfedges.  A thread that cannot be started, for
// want of threads or of memory, is done without; false: out of memory.
inline bool build_lists(const cc_Mesh *const *meshes, std::vector<CageLists> &lists) {
    std::atomic<size_t> next{0};
    std::atomic<bool> ok{true};
    auto work = [&]() {
        try {
            for (size_t i = next++; i < lists.size(); i = next++) {
                build_cage_rings(meshes[i], lists[i].r);
                if (lists[i].r.ok) build_rare_table(meshes[i], lists[i].r, lists[i].rt);
            }
        } catch (const std::bad_alloc &) {
            ok = false;
        }
    };
    int64_t H = 0;
    for (size_t i = 0; i < lists.size(); ++i) H += meshes[i]->halfedgeCount;
    const int64_t threads = std::min<int64_t>({8, (int64_t)lists.size(), (int64_t)std::thread::hardware_concurrency(), H >> 14});
    std::vector<std::thread> pool;
    try {
        pool.reserve(8);
        for (int64_t i = 1; i < threads; ++i) pool.emplace_back(work);
    } catch (const std::exception &) {   // system_error, bad_alloc
    }
    work();
    for (std::thread &t : pool) t.join();
    return ok;
}

}  // namespace cch
