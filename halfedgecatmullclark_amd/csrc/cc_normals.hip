// Per-halfedge normals of the finest level, the step after refinement that
// the reference defines only in its GL shaders
// (glsl/CatmullClark_Scatter.glsl:931-960):
//   corner normal of h  normalize(cross(P(next h) - P(h), P(prev h) - P(h)))
//   vertex normal of h  normalize(corner(h) + the corner normals of the
//                       halfedges met walking it = twin(prev(it)) from h),
//                       or corner(h) when the walk reaches a boundary
// with normalize(v) = v * (1 / sqrt(dot(v, v))), correctly rounded, in the
// shaders' operation order (built with -ffp-contract=off).
//
// Two kernels: tile by tile, one thread per quad, the corner normals and the
// vertex normals of rings that close inside the tile; then the other vertices
// from the corner normals the first stored.  Corner normals alone, and cages
// where a vertex may have several rings (CageRings::simple), take one thread
// per halfedge: vertex by vertex, only the representative's ring would be
// written.
#include <stdio.h>

#include "cc_fan.h"
#include "cc_internal.h"
#include "cc_runtime.h"

using namespace cch;

namespace {

__device__ __forceinline__ P3 sub3(P3 a, P3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ P3 cross3(P3 a, P3 b) {
    return {a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y};
}
__device__ __forceinline__ P3 normalize3(P3 v) {
    const float dd = v.x * v.x + v.y * v.y + v.z * v.z;
    const float inv = 1.0f / sqrtf(dd);
    return mul(v, inv);
}

// corner normals, one thread per halfedge of the level (H a multiple of 4,
// blocks of 256: the four lanes of a quad are live together; workgroups in
// contiguous ranges per XCD, so the points a vertex's quads share meet in
// one L2)
__global__ __launch_bounds__(256) void k_corner_normals(const He *__restrict__ he, const P3 *__restrict__ pts,
                                                        int32_t H, P3 *__restrict__ out) {
    const int32_t h = (int32_t)(xcd_block(blockIdx.x, gridDim.x, 1) * blockDim.x + threadIdx.x);
    const bool live = h < H;
    const int4 x = live ? he_gld(he, h) : make_int4(0, 0, 0, 0);
    const P3 v0 = gld(pts + x.z);
    const P3 v2 = {quad_relf<kQuadNext>(v0.x), quad_relf<kQuadNext>(v0.y), quad_relf<kQuadNext>(v0.z)};
    const P3 v1 = {quad_relf<kQuadPrev>(v0.x), quad_relf<kQuadPrev>(v0.y), quad_relf<kQuadPrev>(v0.z)};
    if (live) out[h] = normalize3(cross3(sub3(v2, v0), sub3(v1, v0)));
}

// One owner per level-d vertex, decided from the child numbering as the
// structural owner test does, except that an edge vertex born at level >= 2
// is owned by child 1 of the larger parent halfedge of its edge (or the
// parent on a boundary): one parent twin read instead of the edge's
// representative descent.  Any owner gives the same fan as a cyclic list.
__device__ __forceinline__ bool normal_owner(int32_t h, int d, const DCage &c, const He *const *levels) {
    const int k = zero_digits(h, d);
    const int32_t q = h >> (2 * k);
    const int lvl = d - k;
    const int digit = q & 3;
    const int32_t p = q >> 2;
    if (digit == 3) return false;
    if (lvl >= 2) {
        if (digit == 2) return (p & 3) == 0;
        const int32_t tw = levels[lvl - 1][p].twin;
        return tw < 0 || p > tw;
    }
    const CageHe x = c.he[p];
    if (digit == 0) return c.v2h[x.vert] == p;
    if (digit == 2) return c.f2h[x.face] == p;
    return c.e2h[x.edge] == p;
}

// Vertex normals of every halfedge of a vertex's fan, from its owner.  The
// fan lists the ring in the walk order twin(prev(x)), so the walk from
// member i visits members i+1, ..., i-1: its normal is
// normalize(c_i + ((0 + c_{i+1}) + ... + c_{i-1})), the per-halfedge walk's
// own sums.  On a boundary every member's walk ends at the boundary and its
// normal is its corner normal.
struct VertexNormalsFn {
    const P3 *corner;
    P3 *out;
    const DCage &c;
    __device__ void operator()(const Fan &f) const {
        const int n = f.n;
        if (f.boundary) {
            for (int i = 0; i < n; ++i) {
                const int32_t r = fan_at(f, c, i);
                out[r] = corner[r];
            }
            return;
        }
        if (n <= 4) {
            int32_t r[4];
            P3 cn[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] = fan_at(f, c, q < n ? q : 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) cn[q] = corner[r[q]];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i >= n) break;
                P3 avg = zero3();
#pragma unroll
                for (int k = 1; k < 4; ++k)
                    if (k < n) avg = add(avg, pick4(cn[0], cn[1], cn[2], cn[3], (i + k) % n));
                out[r[i]] = normalize3(add(cn[i], avg));
            }
            return;
        }
        for (int i = 0; i < n; ++i) {
            const int32_t ri = fan_at(f, c, i);
            P3 avg = zero3();
            for (int k = 1; k < n; ++k) avg = add(avg, corner[fan_at(f, c, (i + k) % n)]);
            out[ri] = normalize3(add(corner[ri], avg));
        }
    }
};

// Corner normals, and vertex normals where the ring of four closes inside a
// tile of N quads (one thread per quad, corner normals in LDS).  Halfedges of
// other rings leave their corner normal in `corner`, and one of each ring,
// normal_owner's, a bit in `mask` for k_vertex_normals_far (a vertex born at
// level 1 leaves one for every child 0, 1 and 2 of its ring: the far kernel
// asks the cage).
// Passing every corner normal through memory took 580 + 1298 us at level 7 of
// the 64 x 32 torus, 134 M halfedges: 1.6 GB written and read back three
// times over by the vertices' quads in different workgroups; what has to
// move is the records, the points and the normals, 4.1 GB.
template <int N>
__global__ __launch_bounds__(N, 8) void k_normal_tiles(const He *__restrict__ he, const P3 *__restrict__ pts, int32_t F,
                                                       int d, P3 *__restrict__ corner, uint64_t *__restrict__ mask,
                                                       P3 *__restrict__ out) {
    // Halfedge k of quad q at k (N + 16) + q: without bank conflicts by quad
    // (written) and by halfedge (read); the steps around the rings conflict
    // (1.5 M cycles a CU at level 8 of the torus, an eighth of the kernel).
    constexpr int kRow = N + 16;
    __shared__ float sc[3][4 * kRow];
    __shared__ uint16_t sr[4 * kRow];   // twin(prev), kOut outside the tile or on a boundary
    constexpr int kOut = 0xffff;
    const int q = (int)threadIdx.x;
    const int32_t base = (int32_t)(xcd_block(blockIdx.x, gridDim.x, 1) * N), p = base + q;
    const bool live = p < F;
    const int32_t g = live ? p : 0;
    int32_t nx[4];
    P3 c[4];
    {
        int4 x[4];
        P3 P[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = he_gld(he, 4 * g + k);
#pragma unroll
        for (int k = 0; k < 4; ++k) P[k] = gld(at3v(pts, x[k].z));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            nx[k] = x[(k + 3) & 3].x;
            c[k] = normalize3(cross3(sub3(P[(k + 1) & 3], P[k]), sub3(P[(k + 3) & 3], P[k])));
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int i = k * kRow + q;
        const uint32_t o = (uint32_t)((nx[k] >> 2) - base);   // a boundary's -1 >> 2 is no quad of the tile
        sr[i] = (uint16_t)(live && nx[k] >= 0 && o < (uint32_t)N ? (nx[k] & 3) * kRow + (int)o : kOut);
        sc[0][i] = c[k].x;
        sc[1][i] = c[k].y;
        sc[2][i] = c[k].z;
    }
    __syncthreads();
    // now a lane per halfedge, so that a wave's stores are consecutive
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int l = k * N + q;
        const int32_t h = 4 * base + l;
        const int i = (l & 3) * kRow + (l >> 2);
        const int r1 = sr[i];
        const int r2 = r1 != kOut ? sr[r1] : kOut;
        const int r3 = r2 != kOut ? sr[r2] : kOut;
        const int r4 = r3 != kOut ? sr[r3] : kOut;
        const bool in = (h >> 2) < F, ring = in && r4 == i && r2 != i;   // four distinct halfedges
        const P3 cn = P3{sc[0][i], sc[1][i], sc[2][i]};
        bool mark = false;
        if (ring) {   // summed in walk order
            P3 avg = zero3();
            avg = add(avg, P3{sc[0][r1], sc[1][r1], sc[2][r1]});
            avg = add(avg, P3{sc[0][r2], sc[1][r2], sc[2][r2]});
            avg = add(avg, P3{sc[0][r3], sc[1][r3], sc[2][r3]});
            *at3(out, h) = normalize3(add(cn, avg));
        } else if (in) {
            *at3(corner, h) = cn;
            const int k2 = 2 * zero_digits(h, d);
            const int digit = (h >> k2) & 3;
            const int32_t pp = h >> (k2 + 2);
            if (2 * (d - 1) == k2) {
                mark = digit != 3;
            } else if (digit == 2) {
                mark = (pp & 3) == 0;
            } else if (digit == 1) {   // the parent's twin, from twin(prev(h)) = 4 next(twin) + 3
                const int32_t nxt = he[qprev(h)].twin;
                mark = nxt < 0 || pp > qprev(nxt >> (k2 + 2));
            }
        }
        const uint64_t m = __ballot(mark);
        if ((q & 63) == 0 && in) mask[h >> 6] = m;
    }
}

struct FarNormalsFn {
    VertexNormalsFn fn;
    const LevelTab &t;
    const LevelPtrs &lp;
    int d;
    __device__ void operator()(int32_t h) const {
        if (zero_digits(h, d) == d - 1 && !normal_owner(h, d, fn.c, lp.he)) return;
        Fan f;
        if (marked_fan(h, d, fn.c, t, lp.he, f) >= 0) fn(f);
    }
};

// the vertices k_normal_tiles marked, WORDS mask words per wave
template <int WORDS>
__global__ __launch_bounds__(256) void k_vertex_normals_far(DCage c, LevelTab t, LevelPtrs lp, int d, int32_t H,
                                                            const uint64_t *__restrict__ mask,
                                                            const P3 *__restrict__ corner, P3 *__restrict__ out) {
    __shared__ LevelTab st;
    __shared__ LevelPtrs slp;
    __shared__ uint16_t list[4][64 * WORDS];
    lds_fill(st, t);
    lds_fill(slp, lp);
    __syncthreads();
    const int32_t wave = (int32_t)(xcd_block(blockIdx.x, gridDim.x, 1) * 4 + (threadIdx.x >> 6));
    mask_group<WORDS>(mask, wave * WORDS, (H + 63) >> 6, list[threadIdx.x >> 6],
                      FarNormalsFn{{corner, out, c}, st, slp, d});
}

// vertex normals from the corner normals, one walk per halfedge
__global__ __launch_bounds__(256) void k_vertex_normals(const He *__restrict__ he, const P3 *__restrict__ corner,
                                                        int32_t H, P3 *__restrict__ out) {
    const int32_t h = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (h >= H) return;
    const P3 n = corner[h];
    P3 avg = zero3();
    int32_t it = he[qprev(h)].twin;
    for (int g = 0; it >= 0 && it != h && g < kWalkCap; ++g) {
        avg = add(avg, corner[it]);
        it = he[qprev(it)].twin;
    }
    out[h] = it < 0 ? n : normalize3(add(n, avg));
}

unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// normals of level D from the mirror's level-D halfedges and points
bool ccd_Subd::normals(P3 *out, bool smooth, hipStream_t st) {
    const int64_t H = n.H[D];
    const He *lhe = he + n.offH[D];
    const P3 *lpts = pts + n.offV[D];
    P3 *corner = out;
    if (smooth) {
        // corner normals, and the tile kernel's bits behind them
        if (!nrm_tmp && hip_failed(hipMalloc(&nrm_tmp, sizeof(P3) * (size_t)H + sizeof(uint64_t) * (size_t)((H + 63) / 64)),
                                   "hipMalloc(corner normals)"))
            return false;
        corner = nrm_tmp;
    }
    if (smooth && D >= 1 && simple) {
        uint64_t *mask = reinterpret_cast<uint64_t *>(nrm_tmp + H);   // H is a multiple of 4: 8-byte aligned
        const int32_t F = (int32_t)(H / 4);
        const bool big = F >= kTileBigFrom;
        const int64_t words = (H + 63) / 64, tile = big ? kTileBig : kTileSmall, per = 4 * (big ? kFarWords : kOwnerWords);
        const dim3 grid((unsigned)((F + tile - 1) / tile)), far((unsigned)((words + per - 1) / per));
        const auto tiles = [&](auto k) {
            hipLaunchKernelGGL(k, grid, dim3((unsigned)tile), 0, st, lhe, lpts, F, D, corner, mask, out);
        };
        const auto rest = [&](auto k) {
            hipLaunchKernelGGL(k, far, dim3(256), 0, st, cage_view(nullptr), tab, level_ptrs(), D, (int32_t)H,
                               (const uint64_t *)mask, (const P3 *)corner, out);
        };
        tiles(big ? k_normal_tiles<kTileBig> : k_normal_tiles<kTileSmall>);
        if (big) rest(k_vertex_normals_far<kFarWords>);
        else rest(k_vertex_normals_far<kOwnerWords>);
    } else {
        hipLaunchKernelGGL(k_corner_normals, dim3(blocks_for(H)), dim3(256), 0, st, lhe, lpts, (int32_t)H, corner);
        if (smooth)
            hipLaunchKernelGGL(k_vertex_normals, dim3(blocks_for(H)), dim3(256), 0, st, lhe, (const P3 *)corner,
                               (int32_t)H, out);
    }
    return !hip_failed(hipGetLastError(), "halfedge normals");
}

namespace {

// the host entry points: the level-maxDepth halfedges and points of the
// subd's host arrays go to its device mirror, the normals come back
void host_normals(const cc_Subd *subd, cc_VertexPoint *normals, bool smooth, const char *fname) {
    clear_error();
    if (!normals) {
        set_error(11, "null normals");
        fprintf(stderr, "cc: %s: null normals\n", fname);
        return;
    }
    ccd_Subd *s = host_mirror(subd);
    if (!s) {
        fprintf(stderr, "cc: %s: %s\n", fname, ccs_LastErrorString());
        return;
    }
    DeviceGuard g(s->device);
    hipStream_t st = s->stream;
    const Counts &n = s->n;
    const int D = s->D;
    const int64_t H = n.H[D];
    if (!s->nrm_out && hip_failed(hipMalloc(&s->nrm_out, sizeof(P3) * (size_t)H), "hipMalloc(normals)")) return;
    if (hip_failed(hipMemcpyAsync(s->he + n.offH[D], subd->halfedges + n.offH[D], sizeof(He) * (size_t)H,
                                  hipMemcpyHostToDevice, st), "upload halfedges") ||
        hip_failed(hipMemcpyAsync(s->pts + n.offV[D], subd->vertexPoints + n.offV[D], sizeof(P3) * (size_t)n.V[D],
                                  hipMemcpyHostToDevice, st), "upload points"))
        return;
    if (!s->normals(s->nrm_out, smooth, st)) return;
    if (hip_failed(hipMemcpyAsync(normals, s->nrm_out, sizeof(P3) * (size_t)H, hipMemcpyDeviceToHost, st),
                   "download normals") ||
        hip_failed(hipStreamSynchronize(st), fname))
        return;
}

}  // namespace

extern "C" {

void ccs_HalfedgeNormals(const cc_Subd *subd, cc_VertexPoint *normals) {
    host_normals(subd, normals, true, "ccs_HalfedgeNormals");
}

void ccs_HalfedgeNormals_Fast(const cc_Subd *subd, cc_VertexPoint *normals) {
    host_normals(subd, normals, false, "ccs_HalfedgeNormals_Fast");
}

int32_t ccd_HalfedgeNormals(ccd_Subd *s, float *devNormals, int32_t smooth, void *stream) {
    clear_error();
    if (!s || !devNormals) {
        set_error(11, "ccd_HalfedgeNormals: null argument");
        return last_error();
    }
    DeviceGuard g(s->device);
    if (!s->normals(reinterpret_cast<P3 *>(devNormals), smooth != 0, (hipStream_t)stream))
        return last_error() ? last_error() : 1;
    return 0;
}

}  // extern "C"
