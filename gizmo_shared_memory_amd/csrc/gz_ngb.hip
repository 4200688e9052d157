// Neighbour searches over the tree (shmem/hydro.cc:37-148, the SNode of tree.h:206-226), for many
// centres at once: every particle within radius_q of centre q (ngb_search), and every gas particle
// whose own kernel reaches centre q although q's does not (ngb_search_reverse, with the node
// hmax of Tree::init_hmax / raise_hmax, tree.cc:286-338).
//
// The forward search is walk_spheres (gz_spheres.h) with a lane per query (below). The reverse
// search takes one wavefront per group of 64 consecutive queries: up to 64 stacked nodes are tested
// at once, one per lane, first against the group's bounding box with the node's hmax (and only if
// it exceeds the group's smallest kernel radius), then with the reference's own node test for
// each query of the group in turn, a node staying only if some query admits it — so the wave walks
// the union of its queries' traversals even when the group straddles a jump of the Morton order.
// Node boxes are the reference's SNode boxes (half side widened for float centres) grown by
// vmax * tau + xpad. The particles of kept leaves are staged through LDS 64 at a time and each lane
// tests its own query against every staged particle with the reference's FP64 expression, so the
// sets are exact. Two passes: counts, then (with the offsets) the sorted slots of each query's
// neighbours, which map to particle indices in Morton order, the reference's traversal order.
#include <cfloat>

#include "gz_features.h"
#include "gz_internal.h"
#include "gz_spheres.h"
#include "gz_wave.h"

namespace gz {

struct NgbArgs {
    const WNode* wn;
    const double* gcx;
    const double* gcy;
    const double* gcz;
    const double* size;
    const float* vmax;
    const float* xpad;
    const double4* src;
    const uint32_t* orderbuf;
    const double *cx, *cy, *cz, *radius;
    int nq, ngroups, root, nclusters;
    int qpw; // queries per wave (a power of two, at most 64)
    double snode_eps, tau;
    int* queue;
    int* stack; // stack_cap ints per wave
    int stack_cap;
    int* status; // bit 0: a stack outgrew stack_cap
    uint32_t* count;     // pass 1: neighbours per query
    const size_t* start; // pass 2: CSR offsets
    uint32_t* slots;     // pass 2: the neighbours' sorted slots
    // node hmax, the gas kernel radii by particle, the gas count
    const float* hmax;
    const double* h;
    size_t n_gas;
};

// The search node's half side (tree.cc:496-506): float-safe, never smaller than the true one.
__device__ __forceinline__ float snode_half(const NgbArgs& a, int i) {
    return snode_half_of(a.gcx[i], a.gcy[i], a.gcz[i], a.size[i], a.snode_eps);
}

// The reverse search (hydro.cc:110-148): radius[q] is the query's own kernel radius h_q, a node is a
// candidate only when its hmax exceeds the smallest h_q of the group, its reach is hmax, and a
// leaf particle j counts when it is gas and h_q <= r < h[j].
template <bool FILL>
__global__ __launch_bounds__(64) void k_ngb_rev(NgbArgs a) {
    __shared__ int s_lpre[64], s_lplo[64]; // kept leaves: first staged index, first slot
    __shared__ double s_px[64], s_py[64], s_pz[64], s_h2[64];
    __shared__ int s_slot[64];
    const int lane = threadIdx.x;
    int* const stk = a.stack + (size_t)blockIdx.x * (size_t)a.stack_cap;
    for (;;) {
        int v = 0;
        if (lane == 0) v = atomicAdd(a.queue, 1);
        const int g = __shfl(v, 0);
        if (g >= a.ngroups) break;
        const int q = g * a.qpw + lane;
        const bool live = lane < a.qpw && q < a.nq;
        double qx = 0, qy = 0, qz = 0, r = 0;
        if (live) {
            qx = a.cx[q]; qy = a.cy[q]; qz = a.cz[q];
            r = a.radius[q];
        }
        const double lo0 = wave_min_d(live ? qx : 1e300), hi0 = wave_max_d(live ? qx : -1e300);
        const double lo1 = wave_min_d(live ? qy : 1e300), hi1 = wave_max_d(live ? qy : -1e300);
        const double lo2 = wave_min_d(live ? qz : 1e300), hi2 = wave_max_d(live ? qz : -1e300);
        const double rmin = wave_min_d(live ? r : 1e300);
        const double r2 = r * r;
        uint32_t found = 0;
        size_t out = live && FILL ? a.start[q] : 0;

        // The roots, one per tree of a forest, form a virtual range that is fed onto the stack
        // whenever it holds less than a batch: a forest of any size then needs no more stack
        // than one tree plus a batch (the lists are sorted afterwards, so the order in which
        // the trees are searched does not matter).
        const int nroots = (a.nclusters > 1) ? a.nclusters : 1;
        int rnext = 0;
        int sp = 0;
        bool overflow = false;
        while (sp > 0 || rnext < nroots) {
            if (sp < 64 && rnext < nroots) {
                const int add = min(64 - sp, nroots - rnext);
                if (lane < add) stk[sp + lane] = (a.nclusters > 1) ? rnext + lane : a.root;
                sp += add;
                rnext += add;
                __threadfence_block();
                __syncthreads();
            }
            const int k = min(sp, 64);
            const int base = sp - k;
            const int node = (lane < k) ? stk[base + lane] : -1;
            sp = base;
            bool keep = false, leaf = false;
            // the node as the per-query test below needs it (kept nodes only)
            double nc0 = 0, nc1 = 0, nc2 = 0, nhalf = 0, nxpad = 0, nvmax = 0, nhm = 0;
            int first = -1, nch = 0, plo = 0, phi = 0;
            if (node >= 0) {
                const WNode w = a.wn[node];
                const float half = snode_half(a, node);
                const double hm = (double)a.hmax[node];
                double dist = hm + (double)half + (double)a.xpad[node];
                if (a.tau > 0) dist += (double)a.vmax[node] * a.tau;
                const double c0 = (double)(float)a.gcx[node], c1 = (double)(float)a.gcy[node],
                             c2 = (double)(float)a.gcz[node];
                const double d0 = fmax(0.0, fmax(lo0 - c0, c0 - hi0));
                const double d1 = fmax(0.0, fmax(lo1 - c1, c1 - hi1));
                const double d2 = fmax(0.0, fmax(lo2 - c2, c2 - hi2));
                if (hm > rmin && d0 <= dist && d1 <= dist && d2 <= dist) {
                    const double ds = dist + 0.7320508075688772 * (double)half;
                    keep = d0 * d0 + d1 * d1 + d2 * d2 <= ds * ds;
                }
                if (keep) {
                    nc0 = c0; nc1 = c1; nc2 = c2;
                    nhalf = (double)half;
                    nxpad = (double)a.xpad[node];
                    nvmax = (double)a.vmax[node];
                    nhm = hm;
                    first = w.first;
                    if (first < 0) {
                        leaf = true;
                        plo = w.plo;
                        phi = w.phi;
                    } else {
                        nch = w.nchild;
                    }
                }
            }
            // A kept node is dropped when the reference's node test (hydro.cc:55-72, reverse
            // :120-133) rejects it for every query of the group: the group's box and largest
            // radius admit it, but no single query needs it (a group that straddles a jump of
            // the Morton order has a wide box). The wave then walks the union of its queries'
            // own traversals.
            {
                uint64_t rem = __ballot(keep), need = 0;
                while (rem) {
                    const int sl = __ffsll((unsigned long long)rem) - 1;
                    rem &= rem - 1;
                    const double b0 = __shfl(nc0, sl), b1 = __shfl(nc1, sl), b2 = __shfl(nc2, sl);
                    const double bh = __shfl(nhalf, sl), bx = __shfl(nxpad, sl);
                    const double bv = __shfl(nvmax, sl), bm = __shfl(nhm, sl);
                    bool hit = false;
                    if (live && bm > r) {
                        double dist = bm + bh + bx;
                        if (a.tau > 0) dist += bv * a.tau;
                        const double dx = b0 - qx, dy = b1 - qy, dz = b2 - qz;
                        if (!(dx > dist || -dx > dist) && !(dy > dist || -dy > dist) &&
                            !(dz > dist || -dz > dist)) {
                            dist += 0.7320508075688772 * bh;
                            hit = !(dx * dx + dy * dy + dz * dz > dist * dist);
                        }
                    }
                    if (__ballot(hit)) need |= 1ull << sl;
                }
                if (!((need >> lane) & 1ull)) {
                    keep = false;
                    leaf = false;
                    nch = 0;
                }
            }
            // children of kept interior nodes go on the stack
            int ctot = 0;
            const int coff = wave_excl_scan(nch, ctot);
            if (sp + ctot > a.stack_cap) {
                overflow = true;
                break;
            }
            for (int c = 0; c < nch; ++c) stk[sp + coff + c] = first + c;
            sp += ctot;
            // Particles of the kept leaves: the wave loads up to 64 at a time, one per lane, into
            // LDS, and every lane then tests its own query against each staged particle.
            const uint64_t lb = __ballot(leaf);
            if (lb) {
                const int nleaf = __popcll(lb);
                int ptot = 0;
                const int poff = wave_excl_scan(leaf ? phi - plo : 0, ptot);
                if (leaf) {
                    const int li = (int)__builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(lb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)lb, 0u));
                    s_lpre[li] = poff;
                    s_lplo[li] = plo;
                }
                __syncthreads();
                for (int base = 0; base < ptot; base += 64) {
                    const int idx = base + lane;
                    if (idx < ptot) {
                        int lo_ = 0, hi_ = nleaf; // the last leaf li with s_lpre[li] <= idx
                        while (hi_ - lo_ > 1) {
                            const int mid = (lo_ + hi_) >> 1;
                            if (s_lpre[mid] <= idx) lo_ = mid;
                            else hi_ = mid;
                        }
                        const int s = s_lplo[lo_] + (idx - s_lpre[lo_]);
                        const double4 p = a.src[s];
                        s_px[lane] = p.x;
                        s_py[lane] = p.y;
                        s_pz[lane] = p.z;
                        s_slot[lane] = s;
                        const uint32_t j = a.orderbuf[s];
                        const double hj = (j < a.n_gas) ? a.h[j] : 0.0;
                        s_h2[lane] = (j < a.n_gas) ? hj * hj : -1.0; // -1: not gas
                    }
                    __syncthreads();
                    const int cnt = min(64, ptot - base);
                    for (int e = 0; e < cnt; ++e) {
                        const double ex = s_px[e] - qx, ey = s_py[e] - qy, ez = s_pz[e] - qz;
                        const double d2 = ex * ex + ey * ey + ez * ez;
                        const bool in = d2 >= r2 && d2 < s_h2[e];
                        if (live && in) {
                            if (FILL) a.slots[out++] = (uint32_t)s_slot[e];
                            ++found;
                        }
                    }
                    __syncthreads();
                }
            }
            __threadfence_block();
            __syncthreads();
        }
        if (overflow) {
            if (lane == 0) atomicOr(a.status, 1);
            continue;
        }
        if (!FILL && live) a.count[q] = found;
    }
}

// The per-query lists of more than kFinishLds neighbours: a Shell sort in place.
__device__ void shell_sort_u32(uint32_t* s, long long n) {
    for (long long gap = n / 2; gap > 0; gap = (gap == 2) ? 1 : gap * 5 / 11) {
        for (long long i = gap; i < n; ++i) {
            const uint32_t v = s[i];
            long long j = i;
            while (j >= gap && s[j - gap] > v) {
                s[j] = s[j - gap];
                j -= gap;
            }
            s[j] = v;
        }
    }
}

// Each query's neighbours in slot (Morton) order, then as particle indices: one wavefront per
// query (a grid-stride loop over the queries). Up to 64 neighbours: a bitonic sort across the
// lanes' registers; up to kFinishLds: a bitonic sort in LDS, each lane taking every 64th element;
// longer lists (rare: a radius far above the local spacing): a Shell sort by one lane.
constexpr int kFinishLds = 1024;

__device__ __forceinline__ uint32_t bitonic_lanes(uint32_t v, int lane) {
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            const uint32_t o = (uint32_t)__shfl_xor((int)v, j);
            const bool up = ((lane & k) == 0);
            const bool lower = ((lane & j) == 0);
            // the lower lane of a pair keeps the smaller value in an ascending block
            v = (lower == up) ? min(v, o) : max(v, o);
        }
    }
    return v;
}

__global__ __launch_bounds__(64) void k_ngb_finish(int nq, const size_t* __restrict__ start,
                                                   uint32_t* __restrict__ slots,
                                                   const uint32_t* __restrict__ orderbuf,
                                                   uint32_t* __restrict__ found) {
    __shared__ uint32_t buf[kFinishLds];
    const int lane = threadIdx.x;
    for (int q = blockIdx.x; q < nq; q += gridDim.x) {
        const size_t b = start[q];
        const int n = (int)(start[q + 1] - b);
        uint32_t* s = slots + b;
        uint32_t* f = found + b;
        if (n <= 64) {
            uint32_t v = (lane < n) ? s[lane] : 0xFFFFFFFFu;
            v = bitonic_lanes(v, lane);
            if (lane < n) f[lane] = orderbuf[v];
        } else if (n <= kFinishLds) {
            int m = 128;
            while (m < n) m <<= 1;
            for (int i = lane; i < m; i += 64) buf[i] = (i < n) ? s[i] : 0xFFFFFFFFu;
            __syncthreads();
            for (int k = 2; k <= m; k <<= 1) {
                for (int j = k >> 1; j > 0; j >>= 1) {
                    // each pair (i, i ^ j) with i < i ^ j is handled by one lane
                    for (int t = lane; t < (m >> 1); t += 64) {
                        const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                        const int l = i | j;
                        const uint32_t x = buf[i], y = buf[l];
                        const bool up = ((i & k) == 0);
                        if ((x > y) == up) {
                            buf[i] = y;
                            buf[l] = x;
                        }
                    }
                    __syncthreads();
                }
            }
            for (int i = lane; i < n; i += 64) f[i] = orderbuf[buf[i]];
            __syncthreads();
        } else if (lane == 0) {
            shell_sort_u32(s, n);
            for (int i = 0; i < n; ++i) f[i] = orderbuf[s[i]];
        }
    }
}

// Some lists too long for the LDS sort: every list sorted at once by a device radix sort of
// (query << 32 | slot) keys, which keeps each query's range of the CSR and does not slow down on
// long lists (lists that all fit the LDS sort are faster in k_ngb_finish; past kFinishLds it
// falls back to a one-lane Shell sort, hundreds of times slower on lists of 10^4-10^5). One wave
// per query writes its keys.
constexpr size_t kRadixFinishMax = size_t(1) << 28; // 24 B of keys and values per pair
__global__ __launch_bounds__(64) void k_ngb_keys(int nq, const size_t* __restrict__ start,
                                                 const uint32_t* __restrict__ slots,
                                                 uint64_t* __restrict__ keys,
                                                 uint32_t* __restrict__ vals) {
    for (int q = blockIdx.x; q < nq; q += gridDim.x) {
        const size_t b = start[q], e = start[q + 1];
        for (size_t i = b + threadIdx.x; i < e; i += 64) {
            keys[i] = ((uint64_t)q << 32) | slots[i];
            vals[i] = 0;
        }
    }
}
__global__ __launch_bounds__(256) void k_ngb_map(size_t n, const uint64_t* __restrict__ keys,
                                                 const uint32_t* __restrict__ orderbuf,
                                                 uint32_t* __restrict__ found) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        found[i] = orderbuf[(uint32_t)keys[i]];
}

__global__ void k_u32_to_size(int n, const uint32_t* __restrict__ in, size_t* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = in[i];
}

// The sum of the per-query counts in 64 bits (the 32-bit scan that makes the offsets would wrap
// past 2^32 - 1 pairs): a grid-stride sum per thread, one atomic per workgroup.
// The largest count too, which picks how the lists are sorted, and behind it how many exceed
// `limit`.
__global__ __launch_bounds__(256) void k_sum_counts(int n, const uint32_t* __restrict__ in,
                                                    unsigned long long* __restrict__ out,
                                                    uint32_t* __restrict__ max_out,
                                                    uint32_t limit) {
    __shared__ unsigned long long ss[4];
    __shared__ uint32_t sm[4], sl[4];
    unsigned long long s = 0;
    uint32_t mx = 0, over = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        s += in[i];
        mx = max(mx, in[i]);
        over += in[i] > limit ? 1 : 0;
    }
    for (int d = 32; d >= 1; d >>= 1) {
        s += (unsigned long long)__shfl_xor((long long)s, d);
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, d));
        over += (uint32_t)__shfl_xor((int)over, d);
    }
    if ((threadIdx.x & 63) == 0) {
        ss[threadIdx.x >> 6] = s;
        sl[threadIdx.x >> 6] = over;
        sm[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 1; k < 4; ++k) {
        s += ss[k];
        mx = max(mx, sm[k]);
        over += sl[k];
    }
    if (s) atomicAdd(out, s);
    if (over) atomicAdd(max_out + 1, over);
    if (mx) atomicMax(max_out, mx);
}

// h rounded up to float, so that the float bound stays one-sided (tree.cc:286-290).
__device__ __forceinline__ float h_as_bound(double h) {
    const float f = (float)h;
    return ((double)f < h) ? nextafterf(f, 1e30f) : f;
}

// ---- the forward search ----------------------------------------------------------------------------
// A lane per query, 64 consecutive queries per wave, on walk_spheres: a query meets its neighbours
// in slot order, which is its list's order. The first launch counts them and keeps the first
// kNgbRow in a row per query, so that a list is found, counted and ordered in one walk; only
// queries with longer lists are walked again, straight into their place in the CSR: by a wave each
// (k_ngb_long) while they are few, else as they were walked first (FILL).
//
// A lane gives up a list that reaches kNgbLane entries per query of its wave, and a wave of its own
// counts and fills it (k_ngb_count, k_ngb_long): alone in its wave, one lane tests a particle at a
// time. With few queries, one to a wave, each takes the whole wave from the start. ms of 1M Hernquist,
// by lanes throughout / so: 300 queries of 133,000 neighbours each 742 / 314, of 27 .22 / .18; 30,000
// of 3,773 715 / 337, of 420 4.2 / 2.8.
constexpr int kNgbRow = 64;
constexpr uint32_t kNgbLane = 64;
// A wave each up to one query in this many. 1M queries, ms a search with a wave each / walked as
// first, by the share of long lists: Hernquist .0015 1.50 / 1.77, .05 2.04 / 2.25, .11 2.50 / 2.55,
// .20 3.10 / 2.86; halo + disk .008 1.59 / 1.96, .07 2.30 / 2.54, .13 2.83 / 2.86, .22 3.52 / 3.17.
constexpr int kNgbFew = 8;
// Rows take at most so many bytes (4,194,304 queries), beyond which every list is walked twice: of 6M
// Hernquist, that many queries take 4.1 ms and one more 6.6 (10.3 for 4.3M with the separate sort).
constexpr size_t kNgbRowsMax = size_t(1) << 30;

struct NgbFwd {
    SphereNodes nodes;
    const double *cx, *cy, *cz, *radius;
    const uint32_t* orderbuf;
    int nq, qpw;
    uint32_t* count;
    uint32_t* rows; // kNgbRow per query, or NULL
    const size_t* start;
    uint32_t* found;
    uint32_t lane_max; // entries from which on a list is a wave's ...
    uint32_t *big, *n_big; // ... and the queries of these
};

template <bool FILL>
__global__ __launch_bounds__(64) void k_ngb_fwd(NgbFwd a) {
    __shared__ SphereLds lds;
    const int lane = threadIdx.x;
    // Block b runs on XCD b % 8: each XCD gets one contiguous share of the queries.
    const int b = blockIdx.x, nb = gridDim.x;
    const int xcd = b & 7, per = nb >> 3, rem = nb & 7;
    const int q = (xcd * per + min(xcd, rem) + (b >> 3)) * a.qpw + lane;
    bool mine = lane < a.qpw && q < a.nq;
    uint32_t* out = nullptr;
    if (FILL) {
        if (mine) {
            const size_t s = a.start[q], n = a.start[q + 1] - s;
            out = a.found + s;
            mine = n > (size_t)(a.rows ? kNgbRow : 0) && n < (size_t)a.lane_max;
        }
        if (__ballot(mine) == 0) return;
    } else if (a.rows && mine) {
        out = a.rows + (size_t)q * kNgbRow;
    }
    double qx = 0, qy = 0, qz = 0, r = 0;
    if (mine) {
        qx = a.cx[q]; qy = a.cy[q]; qz = a.cz[q];
        r = a.radius[q];
    }
    double r2 = mine ? r * r : -1.0;
    const bool asked = mine;
    const uint32_t room = FILL ? 0xFFFFFFFFu : (a.rows ? (uint32_t)kNgbRow : 0u);
    uint32_t n = 0;
    walk_spheres(a.nodes, mine, qx, qy, qz, r, lds, a.orderbuf, [&](int np, auto allowed) {
        auto test = [&](auto ok) {
#pragma unroll 4
            for (int e = 0; e < np; ++e) {
                const double4 p = lds.p[e];
                const double ex = p.x - qx, ey = p.y - qy, ez = p.z - qz;
                if (ex * ex + ey * ey + ez * ez < r2 && ok(e)) {
                    if (n < room) out[n] = lds.id[e];
                    ++n;
                }
            }
        };
        if (allowed.all) test([](int) { return true; });
        else test(allowed);
        if (!FILL && n >= a.lane_max) {
            mine = false;
            r2 = -1.0;
        }
    });
    if (!FILL && asked) {
        a.count[q] = n; // (of a list given up: lane_max or more)
        if (!mine) a.big[atomicAdd(a.n_big, 1u)] = (uint32_t)q;
    }
}

// A wave per query, of a list of them (*n_list) or all (NULL): its count, and its row if there are.
template <bool PACKED>
__global__ __launch_bounds__(64) void k_ngb_count(NgbFwd a, const uint32_t* __restrict__ list,
                                                  const uint32_t* __restrict__ n_list) {
    __shared__ int stk[kSphStack], lpre[64], lplo[64];
    const int n = list ? (int)*n_list : a.nq;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const uint32_t c = list ? list[i] : (uint32_t)i;
        const double qx = a.cx[c], qy = a.cy[c], qz = a.cz[c], r = a.radius[c];
        const double r2 = r * r;
        uint32_t* const row = a.rows ? a.rows + (size_t)c * kNgbRow : nullptr;
        uint32_t found = 0;
        walk_sphere<PACKED>(a.nodes, qx, qy, qz, r, stk, lpre, lplo,
                            [&](bool some, int slot, const double4& p) {
            const double ex = p.x - qx, ey = p.y - qy, ez = p.z - qz;
            const bool in = some && ex * ex + ey * ey + ez * ez < r2;
            const uint64_t im = __ballot(in);
            if (row && found < (uint32_t)kNgbRow) {
                const uint32_t at = found + (uint32_t)lanes_under(im);
                if (in && at < (uint32_t)kNgbRow) row[at] = a.orderbuf[slot];
            }
            found += (uint32_t)__builtin_popcountll(im);
            return true;
        });
        if (threadIdx.x == 0) a.count[c] = found;
    }
}

// The queries with lists longer than a row, in any order. One atomic per 1,024 queries (an atomic on
// the one counter takes its turn of 12 ns: one per wave came to 93 us for 1M queries).
__global__ __launch_bounds__(1024) void k_ngb_longs(int nq, const size_t* __restrict__ start,
                                                    uint32_t* __restrict__ longs,
                                                    uint32_t* __restrict__ n_longs) {
    __shared__ uint32_t s_n, s_at;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const int q = blockIdx.x * 1024 + threadIdx.x;
    const bool is = q < nq && start[q + 1] - start[q] > (size_t)kNgbRow;
    const uint64_t m = __ballot(is);
    int at = 0;
    if ((threadIdx.x & 63) == 0 && m != 0)
        at = (int)atomicAdd(&s_n, (uint32_t)__builtin_popcountll(m));
    at = __builtin_amdgcn_readfirstlane(at);
    __syncthreads();
    if (threadIdx.x == 0 && s_n != 0) s_at = atomicAdd(n_longs, s_n);
    __syncthreads();
    if (is) longs[s_at + at + lanes_under(m)] = (uint32_t)q;
}

// A wave per listed query (of *n_list; NULL: all whose list is no row). They lie among shorter ones:
// with a lane each, the waves that held one or two of them tested every particle of the largest
// sphere in a lane, and the longest lists' waves set the time.
template <bool PACKED>
__global__ __launch_bounds__(64) void k_ngb_long(NgbFwd a, const uint32_t* __restrict__ list,
                                                 const uint32_t* __restrict__ n_list) {
    __shared__ int stk[kSphStack], lpre[64], lplo[64];
    const int n = list ? (int)*n_list : a.nq;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const uint32_t c = list ? list[i] : (uint32_t)i;
        if (a.start[c + 1] - a.start[c] <= (size_t)(a.rows ? kNgbRow : 0)) continue;
        const double qx = a.cx[c], qy = a.cy[c], qz = a.cz[c], r = a.radius[c];
        const double r2 = r * r;
        size_t at = a.start[c];
        walk_sphere<PACKED>(a.nodes, qx, qy, qz, r, stk, lpre, lplo,
                            [&](bool some, int slot, const double4& p) {
            const double ex = p.x - qx, ey = p.y - qy, ez = p.z - qz;
            const bool in = some && ex * ex + ey * ey + ez * ez < r2;
            const uint64_t im = __ballot(in);
            if (in) a.found[at + lanes_under(im)] = a.orderbuf[slot];
            at += __builtin_popcountll(im);
            return true;
        });
    }
}

// The rows into their places: half a wave per query, those with longer lists left to the launches
// above.
__global__ __launch_bounds__(256) void k_ngb_rows(int nq, const size_t* __restrict__ start,
                                                  const uint32_t* __restrict__ rows,
                                                  uint32_t* __restrict__ found) {
    const int lane = threadIdx.x & 31;
    for (int q = blockIdx.x * 8 + (threadIdx.x >> 5); q < nq; q += gridDim.x * 8) {
        const size_t s = start[q];
        const int n = (int)min((size_t)(kNgbRow + 1), start[q + 1] - s);
        if (n > kNgbRow) continue;
        const uint32_t* row = rows + (size_t)q * kNgbRow;
        if (lane < n) found[s + lane] = row[lane];
        if (lane + 32 < n) found[s + lane + 32] = row[lane + 32];
    }
}

// The search nodes, one per tree node.
__global__ __launch_bounds__(256) void k_sphere_nodes(int nn, const WNode* __restrict__ wn,
                                                      const double* __restrict__ gcx,
                                                      const double* __restrict__ gcy,
                                                      const double* __restrict__ gcz,
                                                      const double* __restrict__ size,
                                                      const float* __restrict__ xpad,
                                                      const float* __restrict__ vmax,
                                                      double snode_eps, SRec* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    out[i] = search_node(wn, gcx, gcy, gcz, size, xpad, vmax, snode_eps, i);
}

// Sets *moved when a slot's position (the tree's copy) lies outside its leaf's cell by more than
// tol on some axis.
__global__ __launch_bounds__(256) void k_sphere_moved(size_t nl, const double4* __restrict__ src,
                                                       const int* __restrict__ slot_leaf,
                                                       const double* __restrict__ gcx,
                                                       const double* __restrict__ gcy,
                                                       const double* __restrict__ gcz,
                                                       const double* __restrict__ size, double tol,
                                                       int* __restrict__ moved) {
    const size_t r = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= nl) return;
    const double4 q = src[r];
    const int leaf = slot_leaf[r];
    const double lim = 0.5 * size[leaf] + tol;
    const bool in = fabs(q.x - gcx[leaf]) <= lim && fabs(q.y - gcy[leaf]) <= lim &&
                    fabs(q.z - gcz[leaf]) <= lim; // (false for a NaN)
    if (!in) *moved = 1;
}

gz_status launch_sphere_nodes(const gz_tree* t, double tau, SRec* srec, int* moved,
                              SphereNodes* out, hipStream_t st) {
    const double snode_eps = 1e-6 * t->root_box[3];
    *out = {srec, moved, t->wn, t->gcx, t->gcy, t->gcz, t->size, t->xpad, t->vmax,
            snode_eps, t->src, t->root, t->n_clusters, tau};
    if (!srec) return GZ_OK;
    if (t->nnodes > 0)
        k_sphere_nodes<<<(unsigned)((t->nnodes + 255) / 256), 256, 0, st>>>(
            t->nnodes, t->wn, t->gcx, t->gcy, t->gcz, t->size, t->xpad, t->vmax, snode_eps, srec);
    if (t->n_live > 0)
        k_sphere_moved<<<(unsigned)((t->n_live + 255) / 256), 256, 0, st>>>(
            t->n_live, t->src, t->slot_leaf, t->gcx, t->gcy, t->gcz, t->size, 0.5 * snode_eps,
            moved);
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}

// ---- the reverse search's node hmax ---------------------------------------------------------------
// init_hmax (tree.cc:332-338): each leaf takes the largest rounded-up h of its gas particles (an
// atomic max on the float's bits, which order like the values for h >= 0), then each level from
// the bottom takes the largest of its children's. The reference's per-particle climb with an
// early exit ends with the same subtree maxima.
__global__ __launch_bounds__(256) void k_hmax_leaf(size_t n_live, const uint32_t* __restrict__ orderbuf,
                                                   const int* __restrict__ slot_leaf,
                                                   const double* __restrict__ h, size_t n_hgas,
                                                   unsigned* __restrict__ hbits) {
    const size_t s = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= n_live) return;
    const uint32_t j = orderbuf[s];
    if (j >= n_hgas) return;
    const double hj = h[j];
    const int leaf = slot_leaf[s];
    if (!(hj > 0) || leaf < 0) return;
    atomicMax(&hbits[leaf], __float_as_uint(h_as_bound(hj)));
}

// raise_hmax (tree.cc:293-301) for the leaf of each listed particle: up the ancestors with an
// atomic max on the float bits, stopping where a node already holds as much.
__global__ __launch_bounds__(256) void k_raise_hmax(const uint32_t* __restrict__ idx, size_t n_idx,
                                                    size_t n, const int* __restrict__ leaf_of,
                                                    const int* __restrict__ parent,
                                                    const double* __restrict__ h,
                                                    unsigned* __restrict__ hbits,
                                                    int* __restrict__ status) {
    const size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= n_idx) return;
    const uint32_t i = idx[k];
    if (i >= n) {
        atomicOr(status, 1);
        return;
    }
    const int leaf = leaf_of[i];
    const double hi = h[i];
    if (leaf < 0 || !(hi > 0)) return;
    const unsigned want = __float_as_uint(h_as_bound(hi));
    for (int no = leaf; no >= 0; no = parent[no])
        if (atomicMax(&hbits[no], want) >= want) break;
}

__global__ __launch_bounds__(256) void k_hmax_up(int lo, int hi, const WNode* __restrict__ wn,
                                                 float* __restrict__ hmax) {
    const int n = lo + blockIdx.x * 256 + threadIdx.x;
    if (n >= hi) return;
    const int f = wn[n].first;
    if (f < 0) return;
    float m = 0.f;
    for (int c = f; c < f + wn[n].nchild; ++c) m = fmaxf(m, hmax[c]);
    hmax[n] = m;
}

} // namespace gz

using namespace gz;

namespace {

gz_status ngb_rev_pass(NgbArgs& a, bool fill, int waves, hipStream_t st) {
    GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(a.queue), 2, st));
    const int grid = std::max(1, std::min(waves, a.ngroups));
    if (fill) k_ngb_rev<true><<<grid, 64, 0, st>>>(a);
    else k_ngb_rev<false><<<grid, 64, 0, st>>>(a);
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}
} // namespace

// Both searches.
static gz_status ngb_run(gz_ctx* ctx, const gz_tree* tree, const double* cx, const double* cy,
                         const double* cz, const double* radius, size_t n_q, double tau,
                         size_t* start, uint32_t* found, size_t cap, size_t* total,
                         const double* h, size_t n_gas, bool rev) {
    const char* who = rev ? "gz_tree_ngb_search_reverse" : "gz_tree_ngb_search";
    clear_error();
    if (!ctx || !tree || !total) return fail(GZ_ERR_INVALID, "%s: null argument", who);
    GZ_HIP(hipSetDevice(ctx->device));
    *total = 0;
    if (n_q == 0) return GZ_OK;
    if (!cx || !cy || !cz || !radius || !start)
        return fail(GZ_ERR_INVALID, "%s: null centre, radius or start array", who);
    if (n_q >= 0x7FFFFFFFull) return fail(GZ_ERR_INVALID, "%s: n_q too large", who);
    if (rev && n_gas > 0 && !h) return fail(GZ_ERR_INVALID, "%s: null h", who);
    if (rev && n_gas > tree->n)
        return fail(GZ_ERR_INVALID, "%s: n_gas=%zu exceeds the particle count %zu", who, n_gas,
                    tree->n);
    if (rev && tree->nnodes > 0 && !tree->hmax)
        return fail(GZ_ERR_INVALID, "%s: no node hmax (call gz_tree_init_hmax first)", who);
    hipStream_t st = ctx->stream;
    if (tree->n_live == 0 || tree->nnodes == 0) {
        GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(start), 2 * (n_q + 1), st));
        GZ_HIP(hipStreamSynchronize(st));
        return GZ_OK;
    }
    int* stack = nullptr;
    int stack_cap = 0;
    GZ_TRY(ctx_spill(ctx, &stack, &stack_cap));
    int waves = 0;
    {
        int dev = 0, ncu = 0;
        GZ_HIP(hipGetDevice(&dev));
        GZ_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
        waves = std::max(1, ncu) * 16; // the spill arena holds this many slices
    }
    DevMem& s = ctx->scratch[10];
    ScratchUse s_use(s);
    const size_t cnt_bytes = ((n_q + 1) * sizeof(uint32_t) + 255) & ~size_t(255);
    const size_t big_bytes = rev ? 0 : cnt_bytes;
    const size_t tmp_bytes = (256 + scan_tmp_bytes(n_q + 1) + 255) & ~size_t(255);
    // forward: the search nodes, and a row per query unless the caller has room for more than a row
    // each (such lists would nearly all be walked again; a caller with more room than its lists
    // need walks twice too: 1M of 27 entries 2.2 ms instead of 1.3) (packing reads the whole tree,
    // 75 us at 4M particles: for a few queries it would be most of the search)
    bool packed = !rev && n_q >= tree->n_live / 16;
    size_t srec_bytes = packed ? (size_t)tree->nnodes * sizeof(SRec) : 0;
    const size_t row_bytes = n_q * kNgbRow * sizeof(uint32_t);
    bool rows = !rev && found && cap / kNgbRow <= n_q && row_bytes <= kNgbRowsMax;
    const size_t need = cnt_bytes + tmp_bytes + big_bytes;
    // (both only when there is memory for them)
    rows = rows && s.offer(need + srec_bytes + row_bytes);
    if (packed && !rows && !s.offer(need + srec_bytes)) {
        packed = false;
        srec_bytes = 0;
    }
    GZ_TRY(s.reserve(need));
    uint8_t* b = s.as<uint8_t>();
    uint32_t* count = reinterpret_cast<uint32_t*>(b);
    int* misc = reinterpret_cast<int*>(b + cnt_bytes);
    NgbArgs a{};
    a.wn = tree->wn;
    a.gcx = tree->gcx; a.gcy = tree->gcy; a.gcz = tree->gcz;
    a.size = tree->size;
    a.vmax = tree->vmax;
    a.xpad = tree->xpad;
    a.src = tree->src;
    a.orderbuf = tree->orderbuf;
    a.cx = cx; a.cy = cy; a.cz = cz; a.radius = radius;
    a.nq = (int)n_q;
    // 64 consecutive queries per wave share its traversal; with too few queries to occupy the
    // GPU that way (a small set is often scattered too), fewer per wave, down to one, so that
    // more waves walk at once
    a.qpw = 64;
    while (a.qpw > 1 && (n_q + a.qpw - 1) / a.qpw < (size_t)waves) a.qpw >>= 1;
    a.ngroups = (int)((n_q + a.qpw - 1) / a.qpw);
    a.root = tree->root;
    a.nclusters = tree->n_clusters;
    a.snode_eps = 1e-6 * tree->root_box[3];
    a.tau = tau;
    a.queue = misc;
    a.status = misc + 1;
    a.stack = stack;
    a.stack_cap = stack_cap;
    a.count = count;
    a.hmax = tree->hmax;
    a.h = h;
    a.n_gas = rev ? n_gas : 0;
    GZ_TRY(fill_zero_u32(count, n_q + 1, st));
    unsigned long long* total64 = reinterpret_cast<unsigned long long*>(misc + 4);
    uint32_t* max_count = reinterpret_cast<uint32_t*>(misc + 6);
    GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(total64), 4, st));
    NgbFwd f{};
    const unsigned fgrid = (unsigned)a.ngroups;
    const bool wave_each = a.qpw == 1;
    auto count_by_waves = [&](const uint32_t* list) -> gz_status {
        const unsigned grid = (unsigned)std::min<size_t>(n_q, (size_t)waves);
        if (packed) k_ngb_count<true><<<grid, 64, 0, st>>>(f, list, f.n_big);
        else k_ngb_count<false><<<grid, 64, 0, st>>>(f, list, f.n_big);
        GZ_HIP(hipGetLastError());
        return GZ_OK;
    };
    if (rev) {
        GZ_TRY(ngb_rev_pass(a, false, waves, st));
    } else {
        GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(misc), 9, st));
        GZ_TRY(launch_sphere_nodes(
            tree, tau, packed ? reinterpret_cast<SRec*>(b + need) : nullptr,
            packed ? misc + 8 : nullptr, &f.nodes, st));
        f.cx = cx; f.cy = cy; f.cz = cz; f.radius = radius;
        f.orderbuf = tree->orderbuf;
        f.nq = a.nq;
        f.qpw = a.qpw;
        f.count = count;
        f.rows = rows ? reinterpret_cast<uint32_t*>(b + need + srec_bytes) : nullptr;
        f.start = start;
        f.found = found;
        f.lane_max = kNgbLane * (uint32_t)a.qpw;
        f.big = reinterpret_cast<uint32_t*>(b + cnt_bytes + tmp_bytes);
        f.n_big = reinterpret_cast<uint32_t*>(misc + 3);
        if (wave_each) GZ_TRY(count_by_waves(nullptr));
        else k_ngb_fwd<false><<<fgrid, 64, 0, st>>>(f);
        GZ_HIP(hipGetLastError());
    }
    uint32_t tot32 = 0;
    int h_status = 0;
    unsigned long long h_total = 0;
    uint32_t h_most[2] = {0, 0}; // the longest list, the lists longer than a row
    auto offsets = [&]() -> gz_status {
        k_sum_counts<<<(unsigned)std::min<size_t>(256, (n_q + 255) / 256), 256, 0, st>>>(
            (int)n_q, count, total64, max_count, (uint32_t)kNgbRow);
        GZ_HIP(hipGetLastError());
        // exclusive scan of the counts (count[n_q] = 0 gives the total at start[n_q])
        DevMem& o = ctx->scratch[11];
        GZ_TRY(o.reserve((n_q + 1) * sizeof(uint32_t)));
        GZ_TRY(exclusive_scan_u32(count, o.as<uint32_t>(), n_q + 1, nullptr,
                                  b + cnt_bytes + 256, st));
        k_u32_to_size<<<(unsigned)((n_q + 1 + 255) / 256), 256, 0, st>>>((int)(n_q + 1),
                                                                          o.as<uint32_t>(), start);
        GZ_HIP(hipGetLastError());
        GZ_HIP(hipMemcpyAsync(&tot32, o.as<uint32_t>() + n_q, sizeof tot32,
                              hipMemcpyDeviceToHost, st));
        GZ_HIP(hipMemcpyAsync(h_most, max_count, sizeof h_most, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipMemcpyAsync(&h_status, a.status, sizeof h_status, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipMemcpyAsync(&h_total, total64, sizeof h_total, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        return GZ_OK;
    };
    GZ_TRY(offsets());
    if (!rev && !wave_each && h_most[0] >= f.lane_max) { // some were given up
        GZ_TRY(count_by_waves(f.big));
        GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(total64), 4, st));
        GZ_TRY(offsets());
    }
    if (h_status & 1)
        return fail(GZ_ERR_INTERNAL, "%s: a search stack outgrew %d entries", who,
                    stack_cap);
    const uint32_t h_max = h_most[0], h_long = h_most[1];
    if (h_total > 0xFFFFFFFFull)
        return fail(GZ_ERR_UNSUPPORTED,
                    "%s: %llu neighbour pairs exceed the 2^32 - 1 one call can return; split the "
                    "queries", who, h_total);
    *total = tot32;
    if (!found || cap < (size_t)tot32 || tot32 == 0) return GZ_OK;
    if (!rev) {
        if (rows) {
            k_ngb_rows<<<(unsigned)std::min<size_t>((n_q + 7) / 8, 16384), 256, 0, st>>>(
                (int)n_q, start, f.rows, found);
            GZ_HIP(hipGetLastError());
        }
        auto by_waves = [&](const uint32_t* list, const uint32_t* n_list, size_t most) {
            const unsigned grid = (unsigned)std::min<size_t>(most, (size_t)waves);
            if (packed) k_ngb_long<true><<<grid, 64, 0, st>>>(f, list, n_list);
            else k_ngb_long<false><<<grid, 64, 0, st>>>(f, list, n_list);
        };
        if (wave_each) {
            if (!rows || h_long > 0) by_waves(nullptr, nullptr, n_q);
        } else if (rows && h_long > 0 && h_long <= n_q / kNgbFew) {
            // (the counts are in the offsets: their array takes the list)
            uint32_t* n_longs = reinterpret_cast<uint32_t*>(misc + 2);
            k_ngb_longs<<<(unsigned)((n_q + 1023) / 1024), 1024, 0, st>>>((int)n_q, start, count,
                                                                          n_longs);
            by_waves(count, n_longs, h_long);
        } else if (!rows || h_long > 0) {
            k_ngb_fwd<true><<<fgrid, 64, 0, st>>>(f);
            if (h_max >= f.lane_max) by_waves(f.big, f.n_big, n_q);
        }
        GZ_HIP(hipGetLastError());
        GZ_HIP(hipStreamSynchronize(st));
        return GZ_OK;
    }
    // pass 2: the neighbours' slots, then sorted and mapped to particle indices
    DevMem& sl = ctx->scratch[11];
    GZ_TRY(sl.reserve((size_t)tot32 * sizeof(uint32_t)));
    a.start = start;
    a.slots = sl.as<uint32_t>();
    GZ_TRY(ngb_rev_pass(a, true, waves, st));
    if (h_max > (uint32_t)kFinishLds && (size_t)tot32 <= kRadixFinishMax) {
        DevMem& kb = ctx->scratch[15];
        const size_t nk = tot32;
        GZ_TRY(kb.reserve(nk * (2 * sizeof(uint64_t) + 2 * sizeof(uint32_t))));
        uint64_t* keys = kb.as<uint64_t>();
        uint64_t* keys_alt = keys + nk;
        uint32_t* vals = reinterpret_cast<uint32_t*>(keys_alt + nk);
        uint32_t* vals_alt = vals + nk;
        k_ngb_keys<<<(unsigned)std::min<size_t>(n_q, 65536), 64, 0, st>>>((int)n_q, start,
                                                                        a.slots, keys, vals);
        GZ_HIP(hipGetLastError());
        int qbits = 1;
        while (qbits < 31 && (size_t(1) << qbits) < n_q) ++qbits;
        GZ_TRY(radix_sort_pairs(keys, vals, keys_alt, vals_alt, nk, 32 + qbits, ctx->scratch[3],
                                st));
        k_ngb_map<<<(unsigned)std::min<size_t>((nk + 255) / 256, 65536), 256, 0, st>>>(
            nk, keys, tree->orderbuf, found);
        GZ_HIP(hipGetLastError());
    } else {
        k_ngb_finish<<<(unsigned)std::min<size_t>(n_q, 65536), 64, 0, st>>>(
            (int)n_q, start, a.slots, tree->orderbuf, found);
        GZ_HIP(hipGetLastError());
    }
    GZ_HIP(hipMemcpyAsync(&h_status, a.status, sizeof h_status, hipMemcpyDeviceToHost, st));
    GZ_HIP(hipStreamSynchronize(st));
    if (h_status & 1)
        return fail(GZ_ERR_INTERNAL, "%s: a search stack outgrew %d entries", who,
                    stack_cap);
    return GZ_OK;
}

extern "C" gz_status gz_tree_ngb_search(gz_ctx* ctx, const gz_tree* tree, const double* cx,
                                        const double* cy, const double* cz, const double* radius,
                                        size_t n_q, double tau, size_t* start, uint32_t* found,
                                        size_t cap, size_t* total) {
    return ngb_run(ctx, tree, cx, cy, cz, radius, n_q, tau, start, found, cap, total, nullptr, 0,
                   false);
}

extern "C" gz_status gz_tree_ngb_search_reverse(gz_ctx* ctx, const gz_tree* tree,
                                                const double* h, size_t n_gas, const double* cx,
                                                const double* cy, const double* cz,
                                                const double* h_q, size_t n_q, double tau,
                                                size_t* start, uint32_t* found, size_t cap,
                                                size_t* total) {
    return ngb_run(ctx, tree, cx, cy, cz, h_q, n_q, tau, start, found, cap, total, h, n_gas,
                   true);
}

extern "C" gz_status gz_tree_init_hmax(gz_ctx* ctx, gz_tree* tree, const double* h, size_t n_h,
                                       size_t n_gas) {
    clear_error();
    if (!ctx || !tree) return fail(GZ_ERR_INVALID, "gz_tree_init_hmax: null argument");
    const size_t n_hgas = std::min(n_h, n_gas);
    if (n_hgas > 0 && !h) return fail(GZ_ERR_INVALID, "gz_tree_init_hmax: null h");
    GZ_HIP(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const int nn = tree->nnodes;
    if (nn <= 0) return GZ_OK;
    if (!tree->hmax) {
        void* p = nullptr;
        GZ_TRY(device_alloc(ctx->blocks.get(), &p, (size_t)nn * sizeof(float)));
        tree->hmax = static_cast<float*>(p);
    }
    GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(tree->hmax), (size_t)nn, st));
    if (n_hgas > 0 && tree->n_live > 0) {
        k_hmax_leaf<<<(unsigned)((tree->n_live + 255) / 256), 256, 0, st>>>(
            tree->n_live, tree->orderbuf, tree->slot_leaf, h, n_hgas,
            reinterpret_cast<unsigned*>(tree->hmax));
        GZ_HIP(hipGetLastError());
        // levels bottom-up: children of level L are in level L + 1
        const std::vector<int>& lb = tree->level_begin;
        for (int L = (int)lb.size() - 2; L >= 0; --L) {
            const int lo = lb[L], hi = lb[L + 1];
            if (hi <= lo) continue;
            k_hmax_up<<<(unsigned)((hi - lo + 255) / 256), 256, 0, st>>>(lo, hi, tree->wn,
                                                                         tree->hmax);
            GZ_HIP(hipGetLastError());
        }
    }
    GZ_HIP(hipStreamSynchronize(st));
    return GZ_OK;
}

extern "C" gz_status gz_tree_raise_hmax(gz_ctx* ctx, gz_tree* tree, const uint32_t* idx, size_t n,
                                        const double* h) {
    clear_error();
    if (!ctx || !tree) return fail(GZ_ERR_INVALID, "gz_tree_raise_hmax: null argument");
    if (n == 0) return GZ_OK;
    if (!idx || !h) return fail(GZ_ERR_INVALID, "gz_tree_raise_hmax: null array");
    if (tree->nnodes > 0 && !tree->hmax)
        return fail(GZ_ERR_INVALID, "gz_tree_raise_hmax: no node hmax (call gz_tree_init_hmax first)");
    if (tree->nnodes <= 0) return GZ_OK;
    GZ_HIP(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    DevMem& sm = ctx->scratch[8];
    GZ_TRY(sm.reserve(256));
    int* status = sm.as<int>();
    GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(status), 1, st));
    k_raise_hmax<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(
        idx, n, tree->n, tree->leaf_of, tree->parent, h, reinterpret_cast<unsigned*>(tree->hmax),
        status);
    GZ_HIP(hipGetLastError());
    int hs = 0;
    GZ_HIP(hipMemcpyAsync(&hs, status, sizeof hs, hipMemcpyDeviceToHost, st));
    GZ_HIP(hipStreamSynchronize(st));
    if (hs & 1) return fail(GZ_ERR_INVALID, "gz_tree_raise_hmax: an index is outside the particles");
    return GZ_OK;
}
