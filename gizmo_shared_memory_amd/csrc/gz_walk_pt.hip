// Per-target tree walks on the device: shmem::accel (shmem/tree.cc:528-582) and shmem::potential
// (tree.cc:899-944). Every target meets the tree on its own: a node is accepted or opened by the
// reference's open_node (tree.h:109-144) with the target's own position, softening and aold, an
// accepted node adds its monopole with the spline of the larger softening, and every reached leaf
// (leaves are always opened in these two walks) is summed particle by particle, the target itself
// skipped.
//
// How it runs on CDNA: long target lists, one wavefront takes 64 targets that are neighbours in
// Morton order (fewer when there are too few targets to occupy the GPU that way), one per lane, and
// walks the union of their 64 traversals depth first. The wave visits one node at a
// time; the node's index is wave-uniform, so its 64-byte record comes through the scalar cache
// and every lane still waiting on it tests it against its own target. Lanes that accept it add
// its monopole; the lanes that open it are the mask under which its children are visited. Each
// lane therefore meets exactly the nodes of its own reference traversal and adds the same terms
// (in the same depth-first order); lanes not waiting on a node sit it out. The stack holds
// sibling ranges (next child, children left, lane mask), one per tree level, in lane-indexed
// registers (entry e in lane e, read back with v_readlane): no LDS, and no barrier anywhere. A
// leaf's particles are read once per wave, again through the scalar cache.
//
// Short lists (k_walk_pt1), a wavefront takes one target and tests many of its nodes at a time, in
// the same order.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gz_features.h"
#include "gz_grav_math.h"
#include "gz_internal.h"
#include "gz_wave.h"

namespace gz {

static_assert(kPtDepth >= kMaxLevel + 2, "the range stack must hold one entry per tree level");

// Sort keys of the targets: their sorted slot (n_live for a target outside the tree, so those go
// last), with the list position as the value; tslot as the grouped walk computes it. status bit
// 1: a target index outside the particle set; misc[1] != 0: the list is not in slot order.
__global__ __launch_bounds__(256) void k_pt_keys(const uint32_t* __restrict__ targets, size_t nt,
                                                 const uint32_t* __restrict__ rank,
                                                 const uint32_t* __restrict__ orderbuf,
                                                 size_t n_live, size_t n, int* __restrict__ tslot,
                                                 uint64_t* __restrict__ keys,
                                                 uint32_t* __restrict__ vals,
                                                 int* __restrict__ misc) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nt) return;
    auto slot_of = [&](size_t k) -> uint64_t {
        const uint32_t p = targets[k];
        if (p >= n) return (uint64_t)n_live;
        const uint32_t r = (k < n_live && orderbuf[k] == p) ? (uint32_t)k : rank[p];
        return (r == 0xFFFFFFFFu) ? (uint64_t)n_live : (uint64_t)r;
    };
    if (targets[i] >= n) atomicOr(misc, 2);
    const uint64_t key = slot_of(i);
    tslot[i] = (key == (uint64_t)n_live) ? -1 : (int)key;
    keys[i] = key;
    vals[i] = (uint32_t)i;
    if (i > 0 && slot_of(i - 1) > key) atomicOr(misc + 1, 1);
}

// A pair's term as the factors that a fused multiply-add sums: t0 f, t1 f, t2 f (POT: t0 f). f is 0
// when the two coincide, as a target in the tree and its own particle do exactly (both are read
// from the sorted copy): the reference skips those. Only pairs inside the kernel branch off.
template <bool POT>
__device__ __forceinline__ void pt_pair(const double4 q, double es, double px, double py,
                                        double pz, double pe1, double& t0, double& t1, double& t2,
                                        double& f) {
    const double ex = q.x - px, ey = q.y - py, ez = q.z - pz;
    const double r2 = __builtin_fma(ex, ex, __builtin_fma(ey, ey, ez * ez));
    const double h = dmax_w(pe1, es);
    const double inv = rsqrt_d(r2); // (NaN at 0, where f is not used)
    if (POT) {
        double v = -inv;
        if (r2 < h * h) v = pair_potential_inside(r2, inv, h);
        t0 = q.w;
        f = (r2 > 0) ? v : 0.0;
    } else {
        double v = inv * inv * inv;
        if (r2 < h * h) v = pair_force_over_r_inside(r2, inv, h);
        f = (r2 > 0) ? v * q.w : 0.0;
        t0 = ex;
        t1 = ey;
        t2 = ez;
    }
}

// An accepted node's term in the same form (it lies outside both softenings, open_node's first
// arm, where the spline is exactly Newtonian).
template <bool POT>
__device__ __forceinline__ void pt_node(double dx, double dy, double dz, double mass, bool accept,
                                        double& t0, double& t1, double& t2, double& f) {
    const double r_sq = dx * dx + dy * dy + dz * dz;
    const bool acc = accept & (r_sq > 0);
    const double inv = rsqrt_d(r_sq);
    if (POT) {
        t0 = -mass;
        f = acc ? inv : 0.0;
    } else {
        f = acc ? mass * (inv * inv * inv) : 0.0;
        t0 = dx;
        t1 = dy;
        t2 = dz;
    }
}

// POT: the potential (else the acceleration); REL: per-target aold are given (else the relative
// arm reduces to theta_sq <= 0 for every target, as it does for aold = 0).
template <bool POT, bool REL>
__global__ __launch_bounds__(64) void k_walk_pt(PtArgs a) {
    const int lane = threadIdx.x;
    // Block b runs on XCD b % 8: each XCD gets one contiguous share of the Morton-ordered waves,
    // so its L2 serves one compact region of the tree.
    const int b = blockIdx.x, nb = gridDim.x;
    const int xcd = b & 7, per = nb >> 3, rem = nb & 7;
    const int wv = xcd * per + min(xcd, rem) + (b >> 3);
    const int k = wv * a.tpw + lane;
    const bool valid = lane < a.tpw && k < a.nt;
    int i = 0, my = -1, croot = 0;
    double px = 0, py = 0, pz = 0, pe = 0, ao = 0;
    if (valid) {
        i = a.order ? (int)a.order[k] : k;
        const uint32_t part = a.targets[i];
        my = a.tslot[i];
        if (my >= 0) {
            const double4 q = a.src[my];
            px = q.x; py = q.y; pz = q.z;
            pe = a.src_soft[my];
        } else {
            px = a.x[part]; py = a.y[part]; pz = a.z[part];
            pe = a.soft ? a.soft[part] : 0.0;
        }
        if (REL) ao = a.aold[i];
        croot = root_of(part, a.cluster_start, a.nclusters, a.root);
    }
    const double theta_sq = a.theta_sq;
    const double pe1 = dmax_w(pe, 1e-300); // a pair's kernel extent is max(this, the source's)
    double sx = 0, sy = 0, sz = 0;

    // one pair term for this lane's target
    auto pair = [&](const double4 q, double es) {
        double t0, t1 = 0, t2 = 0, f;
        pt_pair<POT>(q, es, px, py, pz, pe1, t0, t1, t2, f);
        sx = __builtin_fma(t0, f, sx);
        if (!POT) {
            sy = __builtin_fma(t1, f, sy);
            sz = __builtin_fma(t2, f, sz);
        }
    };

    uint64_t todo = __ballot(valid);
    while (todo != 0) {
        // the lanes whose targets lie under one root (a forest has a root per cluster)
        const int r = __builtin_amdgcn_readlane(croot, (int)__builtin_ctzll(todo));
        uint64_t cm = __ballot(valid && croot == r);
        todo &= ~cm;
        // the current sibling range (next node, nodes left, lanes waiting on it) and the stack of
        // the ranges above it: entry e in lane e of stf/stc/stl/sth. A range is pushed only when
        // a node is opened, so the stack holds at most one range per tree level (the host checks
        // the tree's depth against kPtDepth).
        int cf = r, cc = 1, sp = 0;
        int stf = 0, stc = 0, stl = 0, sth = 0;
        for (;;) {
            if (cc == 0) {
                if (sp == 0) break;
                --sp;
                cf = __builtin_amdgcn_readlane(stf, sp);
                cc = __builtin_amdgcn_readlane(stc, sp);
                cm = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(sth, sp) << 32) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readlane(stl, sp);
            }
            const int node = cf;
            ++cf;
            --cc;
            const WNode w = a.wn[node];
            const bool act = (cm >> lane) & 1ull;
            uint64_t om = 0; // the lanes that open an interior node
            if (w.first < 0) {
                // tree.cc:558-570 / :921-931: a reached leaf is summed particle by particle by
                // every waiting lane, the target itself skipped; two particles per step, their
                // records loaded together
                const int phi = w.phi;
                const double4* qp = a.src + w.plo;
                const double* ep = a.src_soft + w.plo;
                int s = w.plo;
                if (act) { // (the lanes that wait on the leaf, once for all its particles)
                    for (; s + 1 < phi; s += 2, qp += 2, ep += 2) {
                        const double4 q0 = qp[0], q1 = qp[1];
                        const double e0 = ep[0], e1 = ep[1];
                        pair(q0, e0);
                        pair(q1, e1);
                    }
                    if (s < phi) pair(qp[0], ep[0]);
                }
            } else {
                // tree.cc:552-557 (accel) and :915-920 (potential): the offset to the node's
                // centre of mass, its squared norm, and open_node with the target's own bounds
                const double dx = w.cx - px, dy = w.cy - py, dz = w.cz - pz;
                const double r_sq = dx * dx + dy * dy + dz * dz;
                const bool open = act & open_node_d(r_sq, (double)w.len, w.s, w.mass,
                                                    (double)w.soft, pe, REL ? ao : 0.0,
                                                    theta_sq, fabs(dx), fabs(dy), fabs(dz));
                double t0, t1 = 0, t2 = 0, f;
                pt_node<POT>(dx, dy, dz, w.mass, act & !open, t0, t1, t2, f);
                sx = __builtin_fma(t0, f, sx);
                if (!POT) {
                    sy = __builtin_fma(t1, f, sy);
                    sz = __builtin_fma(t2, f, sz);
                }
                om = __ballot(open);
            }
            // descend into an opened node: its remaining siblings (if any) wait on the stack
            // below its children. The stack registers change in this one place of the loop.
            const bool down = om != 0;
            const bool mine = down & (lane == sp);
            stf = mine ? cf : stf;
            stc = mine ? cc : stc;
            stl = mine ? (int)(uint32_t)cm : stl;
            sth = mine ? (int)(uint32_t)(cm >> 32) : sth;
            sp += (down && cc > 0) ? 1 : 0;
            if (down) {
                cf = w.first;
                cc = w.nchild;
                cm = om;
            }
        }
    }
    if (valid) {
        a.ax[i] = a.G * sx;
        if (!POT) {
            a.ay[i] = a.G * sy;
            a.az[i] = a.G * sz;
        }
    }
}

// A wavefront per target, for target lists too short to fill the GPU with a lane each. Up to 64
// nodes are tested at a time, from the top of a stack kept in depth-first order: a node that opens
// is replaced in place by its children, an accepted node or a reached leaf stays, marked, until
// it is next in order. The marked entries at the top are then evaluated together, a lane per
// monopole or particle, and their terms added in that order by a lane per component, with the
// fused multiply-adds of k_walk_pt: the sums are its bits. A lane per target walks one node at a
// time, a chain of some 3,000 dependent visits and pairs (1.2 ms for 1,001 targets of 1M).
constexpr int kPtStack = 640; // stack entries; of these a window of one node may need ...
constexpr int kPtSpare = 160; // ... 7 more for each tree level
constexpr int kPtRun = 32;    // marked entries evaluated together, when as many are next in order
static_assert(kPtSpare >= 7 * (kMaxLevel + 2), "a window of one must be able to reach a leaf");

// Lists up to this many targets take a wave each. Both kernels timed (ms, a lane / a wave per target)
// on random and on consecutive targets of 1M Hernquist: 1,000 1.30 / 0.32 and 0.54 / 0.15, 16,384
// 2.72 / 0.73 and 1.10 / 0.74, 32,768 3.02 / 1.26 and 1.37 / 1.49; of 4M halo + disk 16,384 4.32 /
// 1.09 and 1.94 / 1.18, 32,768 5.38 / 1.96 and 2.07 / 2.13.
constexpr int kPtWave = 24576;

template <bool POT, bool REL>
__global__ __launch_bounds__(64) void k_walk_pt1(PtArgs a) {
    __shared__ int s_stk[kPtStack];
    __shared__ int s_pre[64], s_ent[64];
    __shared__ double s_t[4][65]; // POT: the factors of m v; else the offset and the factor
    const int lane = threadIdx.x;
    // XCD-contiguous shares, as k_walk_pt
    const int b = blockIdx.x, nblk = gridDim.x;
    const int xcd = b & 7, per = nblk >> 3, rem = nblk & 7;
    const int k = xcd * per + min(xcd, rem) + (b >> 3);
    const int i = a.order ? (int)a.order[k] : k;
    const uint32_t part = a.targets[i];
    const int my = a.tslot[i];
    double px, py, pz, pe, ao = 0;
    if (my >= 0) {
        const double4 q = a.src[my];
        px = q.x; py = q.y; pz = q.z;
        pe = a.src_soft[my];
    } else {
        px = a.x[part]; py = a.y[part]; pz = a.z[part];
        pe = a.soft ? a.soft[part] : 0.0;
    }
    if (REL) ao = a.aold[i];
    const double pe1 = dmax_w(pe, 1e-300);
    double acc = 0; // lane c < 3 (POT: lane 0): component c

    int sp = 1;
    if (lane == 0) s_stk[0] = root_of(part, a.cluster_start, a.nclusters, a.root);
    while (sp > 0) {
        __syncthreads();
        // the window: the next w entries in order, one per lane; smaller when the stack is nearly
        // full, so that it always has room for their children
        const int w = min(sp, max(1, min(64, (kPtStack - kPtSpare - sp) / 7)));
        int ent = 0;
        if (lane < w) ent = s_stk[sp - 1 - lane];
        const uint64_t mark = __ballot(lane < w && ent < 0);
        const int run = (~mark == 0) ? 64 : (int)__builtin_ctzll(~mark);
        if (run < kPtRun && run < w) {
            int n = 0, first = 0;
            if (lane < w) {
                n = 1;
                if (ent >= 0) {
                    const WNode nd = a.wn[ent];
                    bool open = false;
                    if (nd.first >= 0) {
                        const double dx = nd.cx - px, dy = nd.cy - py, dz = nd.cz - pz;
                        const double r_sq = dx * dx + dy * dy + dz * dz;
                        open = open_node_d(r_sq, (double)nd.len, nd.s, nd.mass, (double)nd.soft,
                                           pe, REL ? ao : 0.0, a.theta_sq, fabs(dx), fabs(dy),
                                           fabs(dz));
                    }
                    if (open) {
                        first = nd.first;
                        n = nd.nchild;
                    } else {
                        ent = ~ent;
                    }
                }
            }
            int total;
            const int off = wave_excl_scan(n, total);
            const int top = sp - w + total - 1;
            __syncthreads();
            if (lane < w && ent < 0) {
                s_stk[top - off] = ent;
            } else {
                for (int j = 0; j < n; ++j) s_stk[top - off - j] = first + j;
            }
            sp = top + 1;
            continue;
        }
        // evaluate the run: entry l's terms are its particles, or its one monopole
        sp -= run;
        int cnt = 0;
        if (lane < run) {
            const WNode nd = a.wn[~ent];
            cnt = (nd.first < 0) ? nd.phi - nd.plo : 1;
        }
        int total;
        const int off = wave_excl_scan(cnt, total);
        const uint64_t some = __ballot(cnt > 0);
        if (cnt > 0) {
            const int li = lanes_under(some);
            s_pre[li] = off;
            s_ent[li] = ~ent;
        }
        __syncthreads();
        const int nent = __builtin_popcountll(some);
        for (int g0 = 0; g0 < total; g0 += 64) {
            const int g = g0 + lane;
            double t0 = 0, t1 = 0, t2 = 0, f = 0;
            if (g < total) {
                int lo = 0, hi = nent; // the last entry li with s_pre[li] <= g
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (s_pre[mid] <= g) lo = mid;
                    else hi = mid;
                }
                const WNode* nd = a.wn + s_ent[lo];
                if (nd->first < 0) {
                    const int s = nd->plo + (g - s_pre[lo]);
                    const double4 q = a.src[s];
                    const double es = a.src_soft[s];
                    pt_pair<POT>(q, es, px, py, pz, pe1, t0, t1, t2, f);
                } else {
                    pt_node<POT>(nd->cx - px, nd->cy - py, nd->cz - pz, nd->mass, true, t0, t1,
                                 t2, f);
                }
            }
            s_t[0][lane] = t0;
            if (!POT) {
                s_t[1][lane] = t1;
                s_t[2][lane] = t2;
            }
            s_t[3][lane] = f;
            __syncthreads();
            const int np = min(64, total - g0);
            if (lane < (POT ? 1 : 3)) {
                // eight entries read together (those past np were written as zeros)
                for (int e0 = 0; e0 < np; e0 += 8) {
                    double u[8], v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        u[j] = s_t[lane][e0 + j];
                        v[j] = s_t[3][e0 + j];
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc = __builtin_fma(u[j], v[j], acc);
                }
            }
            __syncthreads();
        }
    }
    if (lane == 0) a.ax[i] = a.G * acc;
    if (!POT) {
        if (lane == 1) a.ay[i] = a.G * acc;
        if (lane == 2) a.az[i] = a.G * acc;
    }
}

gz_status launch_pt_keys(const uint32_t* targets, size_t nt, const gz_tree* t, size_t n,
                         int* tslot, uint64_t* keys, uint32_t* vals, int* misc, hipStream_t st) {
    if (nt == 0) return GZ_OK;
    k_pt_keys<<<(unsigned)((nt + 255) / 256), 256, 0, st>>>(targets, nt, t->rank, t->orderbuf,
                                                            t->n_live, n, tslot, keys, vals, misc);
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}

gz_status launch_walk_pt(const PtArgs& a, bool potential, hipStream_t st) {
    if (a.nt <= 0) return GZ_OK;
    const bool rel = a.aold != nullptr;
    if (a.nt <= kPtWave) {
        if (potential && rel) k_walk_pt1<true, true><<<a.nt, 64, 0, st>>>(a);
        else if (potential) k_walk_pt1<true, false><<<a.nt, 64, 0, st>>>(a);
        else if (rel) k_walk_pt1<false, true><<<a.nt, 64, 0, st>>>(a);
        else k_walk_pt1<false, false><<<a.nt, 64, 0, st>>>(a);
        GZ_HIP(hipGetLastError());
        return GZ_OK;
    }
    const unsigned grid = (unsigned)((a.nt + a.tpw - 1) / a.tpw);
    if (potential && rel) k_walk_pt<true, true><<<grid, 64, 0, st>>>(a);
    else if (potential) k_walk_pt<true, false><<<grid, 64, 0, st>>>(a);
    else if (rel) k_walk_pt<false, true><<<grid, 64, 0, st>>>(a);
    else k_walk_pt<false, false><<<grid, 64, 0, st>>>(a);
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}

} // namespace gz
