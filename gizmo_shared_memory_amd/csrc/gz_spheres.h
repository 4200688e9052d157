// Searches of many spheres over the tree (shmem/hydro.cc:37-108), a lane per sphere and up to 64 of
// them per wave: the search nodes, and the walk that the density rounds and the neighbour search
// share.
#pragma once

#include "gz_features.h"
#include "gz_internal.h"
#include "gz_wave.h"

namespace gz {

constexpr int kSphStack = 640; // entries of a wave's stack ...
constexpr int kSphSpare = 160; // ... of which a window of one node may need 7 a level
constexpr int kSphRun = 16;    // leaves taken together, when as many are next in order
static_assert(kSphSpare >= 7 * (kMaxLevel + 2), "a window of one must be able to reach a leaf");

// One search node, packed per call. The centre and
// half side are the float search node's (tree.cc:496-506); xpad and vmax as the tree holds them;
// link is the first child, or ~plo for a leaf, and span the child count, or phi for a leaf.
struct alignas(32) SRec {
    float cx, cy, cz, half;
    float xpad, vmax;
    int link, span;
};

// Lane l's value, as a scalar.
__device__ __forceinline__ float lane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The search node of tree node i, from the tree's arrays.
__device__ __forceinline__ SRec search_node(const WNode* wn, const double* gcx, const double* gcy,
                                            const double* gcz, const double* size,
                                            const float* xpad, const float* vmax,
                                            double snode_eps, int i) {
    const WNode w = wn[i];
    SRec r;
    r.cx = (float)gcx[i];
    r.cy = (float)gcy[i];
    r.cz = (float)gcz[i];
    r.half = snode_half_of(gcx[i], gcy[i], gcz[i], size[i], snode_eps);
    r.xpad = xpad[i];
    r.vmax = vmax[i];
    r.link = (w.first >= 0) ? w.first : ~w.plo;
    r.span = (w.first >= 0) ? w.nchild : w.phi;
    return r;
}

// The tree as the searches read it: packed records and whether some particle lies outside its
// build-time cell (*moved), or, for searches too few to pack a whole tree for, the tree's arrays.
struct SphereNodes {
    const SRec* srec; // NULL: from the arrays below
    const int* moved; // NULL: taken as moved
    const WNode* wn;
    const double *gcx, *gcy, *gcz, *size;
    const float *xpad, *vmax;
    double snode_eps;
    const double4* src;
    int root, nclusters;
    double tau;
    __device__ __forceinline__ SRec at(int i) const {
        return srec ? srec[i] : search_node(wn, gcx, gcy, gcz, size, xpad, vmax, snode_eps, i);
    }
};

struct SphereLds {
    // the stack, in depth-first order from its top: nodes still to be tested, and (as ~node)
    // leaves that the spheres' box admits, waiting for the nodes before them
    int stk[kSphStack];
    double4 p[64];           // staged particles, their ids, ...
    uint32_t id[64];
    uint64_t pm[64], lm[64]; // ... and the lanes that may take a particle / a leaf's particles
    int lpre[64], lplo[64];
};

// Which staged particles a lane may take: all of them, or those of the leaves that the
// reference's node test admits for its sphere.
struct SphereAllowed {
    bool all;
    const uint32_t* pm;
    uint32_t bit;
    __device__ __forceinline__ bool operator()(int e) const { return (pm[2 * e] & bit) != 0; }
};

// Walks the tree once for the spheres (qx, qy, qz, h) of the lanes with `mine`, and calls
// chunk(np, allowed) on the particles of the leaves that some sphere may reach, in slot order, up
// to 64 at a time in s.p and s.id (their slots, or ids[slot]). Every lane of the wave calls it; chunk
// may clear a lane's `mine`, whose sphere then keeps no node.
template <class Chunk>
__device__ __forceinline__ void walk_spheres(const SphereNodes& a, bool& mine, double qx, double qy,
                                             double qz, double h, SphereLds& s,
                                             const uint32_t* ids, Chunk&& chunk) {
    const int lane = threadIdx.x & 63;
    // the node test of the forward search for this lane's sphere (hydro.cc:55-72)
    auto admits = [&](float cx, float cy, float cz, float half, float xpad, float vmax) -> bool {
        double dist = h + (double)half + (double)xpad;
        if (a.tau > 0) dist += (double)vmax * a.tau;
        const double dx = (double)cx - qx, dy = (double)cy - qy, dz = (double)cz - qz;
        if (!mine || dx > dist || -dx > dist || dy > dist || -dy > dist || dz > dist || -dz > dist)
            return false;
        const double ds = dist + 0.7320508075688772 * (double)half;
        return !(dx * dx + dy * dy + dz * dz > ds * ds);
    };
    // the same for all spheres at once: the box of their centres, their largest radius (a node
    // that any sphere admits passes: each step is monotone in the bounds). One with a NaN finds
    // nothing, and stays out of them.
    const bool sound = mine && qx == qx && qy == qy && qz == qz && h == h;
    const double lo0 = wave_min_d(sound ? qx : 1e300), hi0 = wave_max_d(sound ? qx : -1e300);
    const double lo1 = wave_min_d(sound ? qy : 1e300), hi1 = wave_max_d(sound ? qy : -1e300);
    const double lo2 = wave_min_d(sound ? qz : 1e300), hi2 = wave_max_d(sound ? qz : -1e300);
    const double hmax = wave_max_d(sound ? h : 0.0);
    // Every particle lies in its build-time cell (or within half the margin that the search nodes
    // have beyond it): then a particle within the radius is in leaves that the node test admits,
    // and the test on distance alone picks the reference's neighbours. Otherwise each leaf's node
    // test is kept per sphere.
    // (A negative radius may be admitted and not reach: it keeps the tests too.)
    const bool fresh = a.moved && *a.moved == 0 && __ballot(mine && h < 0) == 0;
    const SphereAllowed allowed{fresh, reinterpret_cast<const uint32_t*>(s.pm) + (lane >> 5),
                                1u << (lane & 31)};
    int r_next = (a.nclusters > 1) ? 0 : a.root; // a forest's roots in order, up to 64 at a time
    const int r_end = (a.nclusters > 1) ? a.nclusters : a.root + 1;
    int sp = 0;
    for (;;) {
        if (sp == 0) {
            if (r_next == r_end) break;
            sp = min(64, r_end - r_next);
            if (lane < sp) s.stk[sp - 1 - lane] = r_next + lane;
            r_next += sp;
            __syncthreads();
        }
        // the window: the first w nodes in depth-first order, one per lane. Replacing one by its
        // children adds at most 7, so a nearly full stack gets a smaller window; at a window of
        // one it grows by 7 a level at most, which kSphSpare covers.
        const int w = min(sp, max(1, min(64, (kSphStack - kSphSpare - sp) / 7)));
        int ent = 0;
        if (lane < w) ent = s.stk[sp - 1 - lane];
        const uint64_t leaf_m = __ballot(lane < w && ent < 0);
        const int run = (~leaf_m == 0) ? 64 : (int)__builtin_ctzll(~leaf_m);
        if (run < kSphRun && run < w) {
            // test the window's nodes against the spheres' box, the interior ones then for each
            // sphere (a box that straddles a jump of the Morton order admits more than any)
            SRec r{};
            int n = 0; // entries that replace this one
            bool inner = false;
            if (lane < w) {
                if (ent < 0) {
                    n = 1;
                } else {
                    r = a.at(ent);
                    double dist = hmax + (double)r.half + (double)r.xpad;
                    if (a.tau > 0) dist += (double)r.vmax * a.tau;
                    const double c0 = r.cx, c1 = r.cy, c2 = r.cz;
                    const double d0 = fmax(0.0, fmax(lo0 - c0, c0 - hi0));
                    const double d1 = fmax(0.0, fmax(lo1 - c1, c1 - hi1));
                    const double d2 = fmax(0.0, fmax(lo2 - c2, c2 - hi2));
                    const double ds = dist + 0.7320508075688772 * (double)r.half;
                    if (d0 <= dist && d1 <= dist && d2 <= dist &&
                        d0 * d0 + d1 * d1 + d2 * d2 <= ds * ds) {
                        inner = r.link >= 0;
                        if (!inner) {
                            n = 1;
                            ent = ~ent;
                        }
                    }
                }
            }
            for (uint64_t rem = __ballot(inner); rem != 0; rem &= rem - 1) {
                const int l = (int)__builtin_ctzll(rem);
                const bool hit = admits(lane_f(r.cx, l), lane_f(r.cy, l), lane_f(r.cz, l),
                                        lane_f(r.half, l), lane_f(r.xpad, l), lane_f(r.vmax, l));
                if (__ballot(hit) != 0 && lane == l) n = r.span;
            }
            int total;
            const int off = wave_excl_scan(n, total);
            const int top = sp - w + total - 1;
            __syncthreads();
            if (n > 0 && ent < 0) {
                s.stk[top - off] = ent;
            } else {
                for (int j = 0; j < n; ++j) s.stk[top - off - j] = r.link + j;
            }
            sp = top + 1;
            __syncthreads();
            continue;
        }
        // the run of leaves at the top: which spheres admit each, and their particles in slot order
        sp -= run;
        SRec r{};
        if (lane < run) r = a.at(~ent);
        uint64_t mym = fresh ? ~0ull : 0ull;
        for (int l = 0; l < run && !fresh; ++l) {
            const uint64_t m = __ballot(admits(lane_f(r.cx, l), lane_f(r.cy, l), lane_f(r.cz, l),
                                               lane_f(r.half, l), lane_f(r.xpad, l),
                                               lane_f(r.vmax, l)));
            if (lane == l) mym = m;
        }
        const int plo = ~r.link, cnt = (lane < run && mym != 0) ? r.span - plo : 0;
        const uint64_t some = __ballot(cnt > 0);
        if (some == 0) continue;
        int total;
        const int off = wave_excl_scan(cnt, total);
        if (cnt > 0) {
            const int li = lanes_under(some);
            s.lpre[li] = off;
            s.lplo[li] = plo;
            s.lm[li] = mym;
        }
        __syncthreads();
        const int nleaf = __builtin_popcountll(some);
        for (int g0 = 0; g0 < total; g0 += 64) {
            const int g = g0 + lane;
            if (g < total) {
                int lo_ = 0, hi_ = nleaf; // the last leaf li with lpre[li] <= g
                while (hi_ - lo_ > 1) {
                    const int mid = (lo_ + hi_) >> 1;
                    if (s.lpre[mid] <= g) lo_ = mid;
                    else hi_ = mid;
                }
                const int slot = s.lplo[lo_] + (g - s.lpre[lo_]);
                s.p[lane] = a.src[slot];
                s.id[lane] = ids ? ids[slot] : (uint32_t)slot;
                s.pm[lane] = s.lm[lo_];
            }
            __syncthreads();
            chunk(min(64, total - g0), allowed);
            __syncthreads();
        }
    }
}

// Walks the tree for one sphere with the whole wave: up to 64 nodes at a time under the reference's
// own node test, on a stack kept as walk_spheres keeps its. take(have, slot, q) is called by every
// lane on the particles of the admitted leaves, in slot order over the calls and their lanes; the
// walk ends when it returns false. PACKED: a.srec is there.
template <bool PACKED, class Take>
__device__ __forceinline__ void walk_sphere(const SphereNodes& a, double qx, double qy, double qz,
                                            double h, int* stk, int* lpre, int* lplo,
                                            Take&& take) {
    const int lane = threadIdx.x & 63;
    int r_next = (a.nclusters > 1) ? 0 : a.root;
    const int r_end = (a.nclusters > 1) ? a.nclusters : a.root + 1;
    int sp = 0;
    for (;;) {
        __syncthreads();
        if (sp == 0) {
            if (r_next == r_end) break;
            sp = min(64, r_end - r_next);
            if (lane < sp) stk[sp - 1 - lane] = r_next + lane;
            r_next += sp;
            __syncthreads();
        }
        // (the stack, its window and its bound are walk_spheres')
        const int w = min(sp, max(1, min(64, (kSphStack - kSphSpare - sp) / 7)));
        int ent = 0;
        if (lane < w) ent = stk[sp - 1 - lane];
        const uint64_t leaf_m = __ballot(lane < w && ent < 0);
        const int run = (~leaf_m == 0) ? 64 : (int)__builtin_ctzll(~leaf_m);
        if (run < kSphRun && run < w) {
            int n = 0, link = 0;
            if (lane < w && ent < 0) {
                n = 1;
            } else if (lane < w) {
                const SRec r = PACKED ? a.srec[ent] : a.at(ent);
                double dist = h + (double)r.half + (double)r.xpad;
                if (a.tau > 0) dist += (double)r.vmax * a.tau;
                const double dx = (double)r.cx - qx, dy = (double)r.cy - qy,
                             dz = (double)r.cz - qz;
                const double ds = dist + 0.7320508075688772 * (double)r.half;
                if (!(dx > dist || -dx > dist) && !(dy > dist || -dy > dist) &&
                    !(dz > dist || -dz > dist) && !(dx * dx + dy * dy + dz * dz > ds * ds)) {
                    link = r.link;
                    n = (link < 0) ? 1 : r.span;
                    if (link < 0) ent = ~ent;
                }
            }
            int total;
            const int off = wave_excl_scan(n, total);
            const int top = sp - w + total - 1;
            __syncthreads();
            if (n > 0 && ent < 0) {
                stk[top - off] = ent;
            } else {
                for (int j = 0; j < n; ++j) stk[top - off - j] = link + j;
            }
            sp = top + 1;
            continue;
        }
        sp -= run;
        int plo = 0, cnt = 0;
        if (lane < run) {
            const SRec r = PACKED ? a.srec[~ent] : a.at(~ent);
            plo = ~r.link;
            cnt = r.span - plo;
        }
        const uint64_t some = __ballot(cnt > 0);
        int total;
        const int off = wave_excl_scan(cnt, total);
        if (cnt > 0) {
            const int li = lanes_under(some);
            lpre[li] = off;
            lplo[li] = plo;
        }
        __syncthreads();
        const int nleaf = __builtin_popcountll(some);
        for (int g0 = 0; g0 < total; g0 += 64) {
            const int g = g0 + lane;
            int slot = 0;
            double4 q = make_double4(0.0, 0.0, 0.0, 0.0);
            if (g < total) {
                int lo_ = 0, hi_ = nleaf; // the last leaf li with lpre[li] <= g
                while (hi_ - lo_ > 1) {
                    const int mid = (lo_ + hi_) >> 1;
                    if (lpre[mid] <= g) lo_ = mid;
                    else hi_ = mid;
                }
                slot = lplo[lo_] + (g - lpre[lo_]);
                q = a.src[slot];
            }
            if (!take(g < total, slot, q)) return;
        }
    }
}

// t's nodes for a walk; with srec (room for t's nodes) and moved (zero before), packed.
gz_status launch_sphere_nodes(const gz_tree* t, double tau, SRec* srec, int* moved,
                              SphereNodes* out, hipStream_t st);

} // namespace gz
