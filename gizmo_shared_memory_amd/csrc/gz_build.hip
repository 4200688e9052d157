// Tree build on the device: bounding box and root cell, Morton keys, radix sort, level-synchronous
// octree topology, bottom-up node moments and the packed walk nodes.
//
// Follows shmem::build (shmem/tree.cc:350-526) and shmem::build_node (tree.cc:70-197). The
// reference builds recursively with OpenMP tasks and an atomic node counter; here every level of
// the tree is one pass over all nodes of that level, children are allocated by a prefix sum, and
// moments are combined bottom-up one level per launch. The resulting tree is the reference's tree
// node for node (same ranges, same geometric cells, same threaded next[]), numbered level-major.
//
// This file is compiled with -ffp-contract=off: key quantisation and the moment sums must round
// exactly as the reference's do (no fused multiply-add), so keys, topology and every node moment
// are bit-identical to the reference built the same way.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>

#include "gz_internal.h"
#include "gz_wave.h"

namespace gz {

constexpr int kThreads = 256;
// The level table on the device: first nodes of levels 0..kMaxLevel + 2, then the nodes that a
// level which outgrew the arena would have needed.
constexpr int kLevNeed = kMaxLevel + 3;
constexpr int kLevInts = kMaxLevel + 4;

static inline unsigned grid_for(size_t n, int threads = kThreads) {
    return (unsigned)((n + threads - 1) / threads);
}

__device__ __forceinline__ double dmin_(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double dmax_(double a, double b) { return (a < b) ? b : a; }

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = dmin_(v, __shfl_xor(v, d));
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = dmax_(v, __shfl_xor(v, d));
    return v;
}

// ---- bounding box + root cell (tree.cc:361-407) ------------------------------------------------
__global__ __launch_bounds__(kThreads) void k_bbox_partial(const double* __restrict__ x,
                                                           const double* __restrict__ y,
                                                           const double* __restrict__ z,
                                                           const double* __restrict__ m, size_t n,
                                                           double* __restrict__ partial,
                                                           uint32_t* __restrict__ live) {
    double lo0 = 1e300, lo1 = 1e300, lo2 = 1e300, hi0 = -1e300, hi1 = -1e300, hi2 = -1e300;
    uint32_t cnt = 0;
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n;
         i += (size_t)gridDim.x * kThreads) {
        if (!(m[i] > 0)) continue;
        ++cnt;
        const double a = x[i], b = y[i], c = z[i];
        lo0 = dmin_(lo0, a); hi0 = dmax_(hi0, a);
        lo1 = dmin_(lo1, b); hi1 = dmax_(hi1, b);
        lo2 = dmin_(lo2, c); hi2 = dmax_(hi2, c);
    }
    lo0 = wave_min(lo0); lo1 = wave_min(lo1); lo2 = wave_min(lo2);
    hi0 = wave_max(hi0); hi1 = wave_max(hi1); hi2 = wave_max(hi2);
    __shared__ double s[4][6];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) {
        s[w][0] = lo0; s[w][1] = lo1; s[w][2] = lo2; s[w][3] = hi0; s[w][4] = hi1; s[w][5] = hi2;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int k = threadIdx.x;
        double v = s[0][k];
        for (int j = 1; j < 4; ++j) v = (k < 3) ? dmin_(v, s[j][k]) : dmax_(v, s[j][k]);
        partial[(size_t)blockIdx.x * 6 + k] = v;
    }
    for (int d = 32; d >= 1; d >>= 1) cnt += __shfl_xor(cnt, d);
    if (lane == 0) live[(size_t)blockIdx.x * 4 + w] = cnt;
}

// splitmix64 draw in [0,1) for RANDOMIZE_GRAVTREE (tree.cc:381-393)
__device__ double splitmix_unit(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return (double)((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
}

// root[0..3] = centre x, y, z and side; root[4..9] = live bounding box lo, hi; root[10] = the live
// particles. One workgroup (one thread took 270 us over the 1024 partial boxes of a 4M build).
__global__ __launch_bounds__(kThreads) void k_root_cell(const double* __restrict__ partial,
                                                        const uint32_t* __restrict__ live, int nb,
                                                        long long seed, double fx, double fy,
                                                        double fz, double* __restrict__ root) {
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    uint32_t cnt = 0;
    for (int b = threadIdx.x; b < nb; b += kThreads)
        for (int k = 0; k < 3; ++k) {
            lo[k] = dmin_(lo[k], partial[(size_t)b * 6 + k]);
            hi[k] = dmax_(hi[k], partial[(size_t)b * 6 + 3 + k]);
        }
    for (int b = threadIdx.x; b < 4 * nb; b += kThreads) cnt += live[b];
    __shared__ double s[4][6];
    __shared__ uint32_t sc[4];
    const int w = threadIdx.x >> 6;
    for (int d = 32; d >= 1; d >>= 1) cnt += __shfl_xor(cnt, d);
    for (int k = 0; k < 3; ++k) {
        lo[k] = wave_min(lo[k]);
        hi[k] = wave_max(hi[k]);
    }
    if ((threadIdx.x & 63) == 0) {
        for (int k = 0; k < 3; ++k) {
            s[w][k] = lo[k];
            s[w][3 + k] = hi[k];
        }
        sc[w] = cnt;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int j = 1; j < 4; ++j) {
        for (int k = 0; k < 3; ++k) {
            lo[k] = dmin_(lo[k], s[j][k]);
            hi[k] = dmax_(hi[k], s[j][3 + k]);
        }
        cnt += sc[j];
    }
    root[10] = (double)cnt;
    double cx = 0.5 * (lo[0] + hi[0]), cy = 0.5 * (lo[1] + hi[1]), cz = 0.5 * (lo[2] + hi[2]);
    double side = dmax_(hi[0] - lo[0], dmax_(hi[1] - lo[1], hi[2] - lo[2])) * 1.0000001;
    if (side <= 0) side = 1.0;
    if (seed >= 0) {
        uint64_t s = (uint64_t)seed * 0x9E3779B97F4A7C15ull;
        cx += side * (splitmix_unit(s) - 0.5);
        cy += side * (splitmix_unit(s) - 0.5);
        cz += side * (splitmix_unit(s) - 0.5);
        side *= 2.0;
    }
    if (fx != 0.0 || fy != 0.0 || fz != 0.0) { // the reference's SHMEM_TREE_SHIFT (tree.cc:400-407)
        cx += fx * side; cy += fy * side; cz += fz * side;
        side *= 1.0 + 2.0 * (fabs(fx) + fabs(fy) + fabs(fz));
    }
    root[0] = cx; root[1] = cy; root[2] = cz; root[3] = side;
    for (int k = 0; k < 3; ++k) { root[4 + k] = lo[k]; root[7 + k] = hi[k]; }
}

// ---- independent clusters (a forest) -------------------------------------------------------------
// Cluster c is particles [cstart[c], cstart[c+1]); each gets its own root cell from its own live
// bounding box, exactly as the single-tree root (tree.cc:361-372), and its own tree.
__device__ __forceinline__ int cluster_of(uint32_t i, const uint32_t* __restrict__ cstart, int nc) {
    int lo = 0, hi = nc; // last c with cstart[c] <= i
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cstart[mid] <= i) lo = mid;
        else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(kThreads) void k_bbox_clusters(const double* __restrict__ x,
                                                            const double* __restrict__ y,
                                                            const double* __restrict__ z,
                                                            const double* __restrict__ m,
                                                            const uint32_t* __restrict__ cstart,
                                                            double* __restrict__ roots) {
    const int c = blockIdx.x;
    double lo0 = 1e300, lo1 = 1e300, lo2 = 1e300, hi0 = -1e300, hi1 = -1e300, hi2 = -1e300;
    for (uint32_t i = cstart[c] + threadIdx.x; i < cstart[c + 1]; i += kThreads) {
        if (!(m[i] > 0)) continue;
        lo0 = dmin_(lo0, x[i]); hi0 = dmax_(hi0, x[i]);
        lo1 = dmin_(lo1, y[i]); hi1 = dmax_(hi1, y[i]);
        lo2 = dmin_(lo2, z[i]); hi2 = dmax_(hi2, z[i]);
    }
    lo0 = wave_min(lo0); lo1 = wave_min(lo1); lo2 = wave_min(lo2);
    hi0 = wave_max(hi0); hi1 = wave_max(hi1); hi2 = wave_max(hi2);
    __shared__ double s[4][6];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) {
        s[w][0] = lo0; s[w][1] = lo1; s[w][2] = lo2; s[w][3] = hi0; s[w][4] = hi1; s[w][5] = hi2;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    double lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = s[0][k];
        hi[k] = s[0][3 + k];
        for (int j = 1; j < 4; ++j) {
            lo[k] = dmin_(lo[k], s[j][k]);
            hi[k] = dmax_(hi[k], s[j][3 + k]);
        }
    }
    double side = dmax_(hi[0] - lo[0], dmax_(hi[1] - lo[1], hi[2] - lo[2])) * 1.0000001;
    if (side <= 0) side = 1.0;
    double* r = roots + (size_t)c * 4;
    r[0] = 0.5 * (lo[0] + hi[0]);
    r[1] = 0.5 * (lo[1] + hi[1]);
    r[2] = 0.5 * (lo[2] + hi[2]);
    r[3] = side;
}

__global__ __launch_bounds__(kThreads) void k_cluster_keys(const uint32_t* __restrict__ v,
                                                           size_t nl,
                                                           const uint32_t* __restrict__ cstart,
                                                           int nc, uint64_t* __restrict__ ck) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r < nl) ck[r] = (uint64_t)cluster_of(v[r], cstart, nc);
}

__global__ __launch_bounds__(kThreads) void k_cluster_counts(const uint32_t* __restrict__ v,
                                                             size_t nl,
                                                             const uint32_t* __restrict__ cstart,
                                                             int nc, int* __restrict__ cnt) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r < nl) atomicAdd(&cnt[cluster_of(v[r], cstart, nc)], 1);
}

__global__ __launch_bounds__(kThreads) void k_init_roots(int nc, const double* __restrict__ roots,
                                                         const int* __restrict__ rstart, int* nlo,
                                                         int* nhi, double* gcx, double* gcy,
                                                         double* gcz, double* size, int* parent,
                                                         int* next, int* lev) {
    const int c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= nc) return;
    if (c == 0) {
        lev[0] = 0;
        lev[1] = nc;
        lev[kLevNeed] = 0;
    }
    nlo[c] = rstart[c];
    nhi[c] = rstart[c + 1];
    gcx[c] = roots[4 * c];
    gcy[c] = roots[4 * c + 1];
    gcz[c] = roots[4 * c + 2];
    size[c] = roots[4 * c + 3];
    parent[c] = -1;
    next[c] = -1;
}

// ---- live filter + keys (tree.cc:355-359, 409-418) ----------------------------------------------
__global__ __launch_bounds__(kThreads) void k_live_flags(const double* __restrict__ m, size_t n,
                                                         uint32_t* __restrict__ flag) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n) flag[i] = (m[i] > 0) ? 1u : 0u;
}

__global__ __launch_bounds__(kThreads) void k_live_compact(const double* __restrict__ m, size_t n,
                                                           const uint32_t* __restrict__ pos,
                                                           uint32_t* __restrict__ order) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n && m[i] > 0) order[pos[i]] = (uint32_t)i;
}

__device__ __forceinline__ uint64_t spread3(uint32_t v) {
    uint64_t x = v & 0x1FFFFFu;
    x = (x | (x << 32)) & 0x1F00000000FFFFull;
    x = (x | (x << 16)) & 0x1F0000FF0000FFull;
    x = (x | (x << 8)) & 0x100F00F00F00F00Full;
    x = (x | (x << 4)) & 0x10C30C30C30C30C3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

__global__ __launch_bounds__(kThreads) void k_keys(const uint32_t* __restrict__ order, size_t nl,
                                                   const double* __restrict__ x,
                                                   const double* __restrict__ y,
                                                   const double* __restrict__ z,
                                                   const double* __restrict__ roots,
                                                   const uint32_t* __restrict__ cstart, int nc,
                                                   uint64_t* __restrict__ keys,
                                                   uint32_t* __restrict__ vals) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= nl) return;
    const uint32_t i = order ? order[r] : (uint32_t)r;
    if (!order) vals[r] = i;
    const double* root = roots + (nc > 1 ? (size_t)cluster_of(i, cstart, nc) * 4 : 0);
    const double side = root[3];
    const double scale = (double)((1u << kMaxLevel) - 1) / side;
    const double bx = root[0] - 0.5 * side, by = root[1] - 0.5 * side, bz = root[2] - 0.5 * side;
    const uint32_t a = (uint32_t)((x[i] - bx) * scale);
    const uint32_t b = (uint32_t)((y[i] - by) * scale);
    const uint32_t c = (uint32_t)((z[i] - bz) * scale);
    keys[r] = spread3(a) | (spread3(b) << 1) | (spread3(c) << 2);
}

// One particle's sources in a line of their own.
struct alignas(64) PRec {
    double x, y, z, m, soft, pad[3];
};

// Sorted copy of the source data (tree.cc:483-485). The particles are read in random order: from
// the caller's arrays that is five partly used lines each, 470 us for 4M particles and bound by
// them. Large sets are therefore first packed to a line per particle (k_pack_rec, a streaming
// pass), which the gather then reads whole: 4M together 235 us. Below kPackRec particles the
// arrays stay in cache and the direct gather is as fast with a launch less.
constexpr size_t kPackRec = size_t(1) << 19;
__global__ __launch_bounds__(kThreads) void k_pack_rec(size_t n, const double* __restrict__ x,
                                                       const double* __restrict__ y,
                                                       const double* __restrict__ z,
                                                       const double* __restrict__ m,
                                                       const double* __restrict__ soft,
                                                       PRec* __restrict__ rec) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    double4* o = reinterpret_cast<double4*>(rec + i);
    o[0] = make_double4(x[i], y[i], z[i], m[i]);
    o[1] = make_double4(soft ? soft[i] : 0.0, 0.0, 0.0, 0.0);
}

__global__ __launch_bounds__(kThreads) void k_gather_rec(const uint32_t* __restrict__ orderbuf,
                                                         size_t nl, const PRec* __restrict__ rec,
                                                         double4* __restrict__ src,
                                                         double* __restrict__ src_soft) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= nl) return;
    const double4* p = reinterpret_cast<const double4*>(rec + orderbuf[r]);
    src[r] = p[0];
    if (src_soft) src_soft[r] = p[1].x;
}

__global__ __launch_bounds__(kThreads) void k_gather_sorted(
    const uint32_t* __restrict__ orderbuf, size_t nl, const double* __restrict__ x,
    const double* __restrict__ y, const double* __restrict__ z, const double* __restrict__ m,
    const double* __restrict__ soft, double4* __restrict__ src, double* __restrict__ src_soft) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= nl) return;
    const uint32_t p = orderbuf[r];
    src[r] = make_double4(x[p], y[p], z[p], m[p]);
    if (src_soft) src_soft[r] = soft ? soft[p] : 0.0;
}

// grow: the records' memory may be allocated (else they are used only if there is room already).
// A line per particle is much to ask for late in a large build: without it the arrays are read.
static gz_status gather_sources(const gz_particles* p, const uint32_t* orderbuf, size_t nl,
                                double4* src, double* src_soft, DevMem& mem, bool grow,
                                hipStream_t st) {
    if (nl == 0) return GZ_OK;
    const size_t rec_bytes = p->n * sizeof(PRec);
    // (packing the dead particles of a set that is mostly dead would cost more than it saves)
    if (nl >= kPackRec && nl >= p->n / 2 &&
        (grow ? mem.offer(rec_bytes) : mem.bytes >= rec_bytes)) {
        k_pack_rec<<<grid_for(p->n), kThreads, 0, st>>>(p->n, p->x, p->y, p->z, p->m, p->soft,
                                                        mem.as<PRec>());
        k_gather_rec<<<grid_for(nl), kThreads, 0, st>>>(orderbuf, nl, mem.as<PRec>(), src,
                                                        src_soft);
    } else {
        k_gather_sorted<<<grid_for(nl), kThreads, 0, st>>>(orderbuf, nl, p->x, p->y, p->z, p->m,
                                                           p->soft, src, src_soft);
    }
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}

gz_status gather_live(gz_ctx* ctx, const gz_particles* p, const gz_tree* t, double4* out) {
    return gather_sources(p, t->orderbuf, t->n_live, out, nullptr, ctx->scratch[2], true,
                          ctx->stream);
}

// The inverse permutation and each particle's leaf, from the sorted side.
__global__ __launch_bounds__(kThreads) void k_particle_links(const uint32_t* __restrict__ orderbuf,
                                                             const int* __restrict__ slot_leaf,
                                                             size_t nl,
                                                             uint32_t* __restrict__ rank,
                                                             int* __restrict__ leaf_of) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= nl) return;
    const uint32_t p = orderbuf[r];
    rank[p] = (uint32_t)r;
    leaf_of[p] = slot_leaf[r];
}

// Sorted copy of the build-time velocities.
__global__ __launch_bounds__(kThreads) void k_gather_vel(const uint32_t* __restrict__ orderbuf,
                                                         size_t nl, const double* __restrict__ vx,
                                                         const double* __restrict__ vy,
                                                         const double* __restrict__ vz,
                                                         double4* __restrict__ svel) {
    const size_t r = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (r >= nl) return;
    const uint32_t p = orderbuf[r];
    svel[r] = make_double4(vx[p], vy[p], vz[p], 0.0);
}

__global__ __launch_bounds__(kThreads) void k_fill_u32(uint32_t* __restrict__ a, size_t n,
                                                       uint32_t v) {
    const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (i < n) a[i] = v;
}

__global__ void k_init_root(const double* __restrict__ root, int nl, int* nlo, int* nhi,
                            double* gcx, double* gcy, double* gcz, double* size, int* parent,
                            int* next, int* lev) {
    lev[0] = 0;
    lev[1] = 1;
    lev[kLevNeed] = 0;
    nlo[0] = 0;
    nhi[0] = nl;
    gcx[0] = root[0];
    gcy[0] = root[1];
    gcz[0] = root[2];
    size[0] = root[3];
    parent[0] = -1;
    next[0] = -1;
}

// ---- topology, two launches per level (tree.cc:86-143) ------------------------------------------
// The level table lev (node ids [lev[L], lev[L+1]) are level L) is kept on the device, so levels
// are enqueued without the host reading a count back in between (16 read-backs of 20 us in a 4M
// build); launches are sized by an upper bound and step over the nodes there are.
constexpr int kLevelChunk = 64; // nodes whose children k_split counts together

// Each node of the level: leaf test, then the start of each octant's run of keys (keys in a node
// share every higher digit, so the 3-bit digit is sorted). Eight lanes take one node, lane o
// finding octant o by binary search; with WIDE a wave takes one node, eight lanes to an octant,
// each step probing eight places at once, for the few nodes of the top levels, whose searches
// would otherwise be 22 dependent loads long (65 us a level at 4M particles by one thread a node).
template <bool WIDE>
__global__ __launch_bounds__(kThreads) void k_split(int level, const int* __restrict__ lev,
                                                    const int* __restrict__ nlo,
                                                    const int* __restrict__ nhi,
                                                    const uint64_t* __restrict__ skey,
                                                    int* __restrict__ oct_start,
                                                    uint32_t* __restrict__ nkids,
                                                    uint32_t* __restrict__ chunk_sum) {
    constexpr int kLanes = WIDE ? 64 : 8;
    constexpr int kPer = kThreads / kLanes; // nodes a workgroup holds at once
    __shared__ uint32_t s_sum[kThreads / kWave];
    const int lb = lev[level], count = lev[level + 1] - lb;
    const int lane = threadIdx.x & 63;
    const int o = WIDE ? (lane >> 3) : (threadIdx.x & 7), probe = lane & 7;
    for (int c0 = blockIdx.x * kLevelChunk; c0 < count; c0 += gridDim.x * kLevelChunk) {
        uint32_t sum = 0; // children of this wave's nodes
        for (int k = 0; k < kLevelChunk && c0 + k < count; k += kPer) {
            const int i = c0 + k + (int)threadIdx.x / kLanes;
            const bool live = i < count;
            int lo = 0, hi = 0;
            if (live) {
                lo = nlo[lb + i];
                hi = nhi[lb + i];
            }
            const bool split = hi - lo > kLeafMax && level < kMaxLevel;
            const int shift = 3 * (kMaxLevel - level - 1);
            int a = lo, b = hi; // the first index in [lo, hi) with digit >= o, or hi, is in [a, b]
            if (!split || o == 0) b = a;
            if (WIDE) {
                while (__ballot(a < b)) {
                    // eight probes from a on cut [a, b) into eight parts; digits ascend, so the
                    // probes below o come first
                    const long long len = b - a;
                    const int at = a + (int)((len * probe) >> 3);
                    const bool below = a < b && (int)((skey[at] >> shift) & 7ull) < o;
                    const uint64_t m = (__ballot(below) >> (lane & 56)) & 0xffull;
                    const int nbelow = __popcll(m);
                    if (a < b) {
                        if (nbelow < 8) b = a + (int)((len * nbelow) >> 3);
                        if (nbelow > 0) a = a + (int)((len * (nbelow - 1)) >> 3) + 1;
                    }
                }
            } else {
                while (a < b) {
                    const int mid = a + ((b - a) >> 1);
                    if ((int)((skey[mid] >> shift) & 7ull) < o) a = mid + 1;
                    else b = mid;
                }
            }
            int e = __shfl_down(a, WIDE ? 8 : 1); // the next octant's start
            if (o == 7) e = hi;
            const uint64_t m = __ballot(split && e > a && (!WIDE || probe == 0));
            if (split && (!WIDE || probe == 0)) oct_start[(size_t)i * 8 + o] = a;
            const uint32_t nk = WIDE ? (uint32_t)__popcll(m)
                                     : (uint32_t)__popcll((m >> (lane & 56)) & 0xffull);
            if (live && (WIDE ? lane == 0 : o == 0)) nkids[i] = nk;
            sum += (uint32_t)__popcll(m);
        }
        if (lane == 0) s_sum[threadIdx.x >> 6] = sum;
        __syncthreads();
        if (threadIdx.x == 0)
            chunk_sum[c0 / kLevelChunk] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
        __syncthreads();
    }
}

// The chunk counts of a level as their exclusive prefix sums, and their total behind them. One
// workgroup, 8,192 counts at a time.
__global__ __launch_bounds__(1024) void k_chunk_scan(int level, const int* __restrict__ lev,
                                                     uint32_t* __restrict__ chunk_sum) {
    constexpr int kEach = 8;
    __shared__ uint32_t s_w[16];
    const int count = lev[level + 1] - lev[level];
    const int nchunk = (count + kLevelChunk - 1) / kLevelChunk;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t carry = 0;
    for (int base = 0; base < nchunk; base += 1024 * kEach) {
        const int i0 = base + (int)threadIdx.x * kEach;
        uint32_t v[kEach], sum = 0;
#pragma unroll
        for (int j = 0; j < kEach; ++j) {
            v[j] = (i0 + j < nchunk) ? chunk_sum[i0 + j] : 0u;
            sum += v[j];
        }
        const uint32_t inc = wave_incl_scan_dpp(sum);
        if (lane == 63) s_w[w] = inc;
        __syncthreads();
        uint32_t off = 0, all = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            off += (k < w) ? s_w[k] : 0u;
            all += s_w[k];
        }
        uint32_t run = carry + off + inc - sum;
#pragma unroll
        for (int j = 0; j < kEach; ++j) {
            if (i0 + j < nchunk) chunk_sum[i0 + j] = run;
            run += v[j];
        }
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) chunk_sum[nchunk] = carry;
}

// Allocate each node's children after the level's own nodes, by the prefix sum of the counts, in
// octant order, with the child cell from halving the parent's (tree.cc:101, 116-118) and the
// threaded successor (tree.cc:340-348): the next sibling, or the parent's successor for the last
// child. A workgroup adds up the chunk counts before its own. Eight lanes write one node's
// children, so neighbouring lanes write neighbouring nodes. When the children would outgrow the
// arena, nothing is emitted, the next level stays empty and lev[kLevNeed] tells the nodes needed.
// A workgroup emits CHUNKS chunks at a time: four where a level may be large (each step adds up the
// level's chunk counts), one in small trees, whose levels are a few steps long. With SCANNED the
// counts are prefix sums already, a launch more for each level; adding them up in each step is
// quadratic in a level's nodes. The levels together, added up / scanned, ms: 4M Hernquist .604 / .624,
// 16.8M .936 / .930, uniform .611 / .541; 33.6M 1.56 / 1.40, uniform 2.42 / 1.21; 67M 3.02 / 2.10,
// uniform 8.54 / 1.96 (with an arena of 3 nodes for 8 particles).
constexpr int kEmitSmall = 1 << 18; // arenas up to this many nodes count as small
constexpr int kEmitScan = 1 << 22;  // from here on the counts are scanned
template <int CHUNKS, bool SCANNED>
__global__ __launch_bounds__(kThreads) void k_emit(
    int level, int cap, int* __restrict__ lev, const uint32_t* __restrict__ nkids,
    const uint32_t* __restrict__ chunk_sum, const int* __restrict__ oct_start,
    int* __restrict__ nlo, int* __restrict__ nhi, double* __restrict__ gcx,
    double* __restrict__ gcy, double* __restrict__ gcz, double* __restrict__ size,
    int* __restrict__ parent, int* __restrict__ next, WNode* __restrict__ wn) {
    constexpr int kNodes = CHUNKS * kLevelChunk;
    static_assert(kNodes <= kThreads, "the prefix of a step is at most one value per thread");
    __shared__ uint32_t s_red[8];
    __shared__ int s_off[kNodes];
    const int lb = lev[level], le = lev[level + 1], count = le - lb;
    const int nchunk = (count + kLevelChunk - 1) / kLevelChunk;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int n0 = blockIdx.x * kNodes; n0 < count || (blockIdx.x == 0 && n0 == 0);
         n0 += gridDim.x * kNodes) {
        // children of the chunks before this step's first, and of all of them
        uint32_t before = 0, all = 0;
        if (SCANNED) {
            before = chunk_sum[n0 / kLevelChunk];
            all = chunk_sum[nchunk];
        } else {
            for (int c = threadIdx.x; c < nchunk; c += kThreads) {
                const uint32_t v = chunk_sum[c];
                before += (c < n0 / kLevelChunk) ? v : 0u;
                all += v;
            }
            for (int d = 32; d >= 1; d >>= 1) {
                before += __shfl_xor(before, d);
                all += __shfl_xor(all, d);
            }
            if (lane == 0) {
                s_red[w] = before;
                s_red[4 + w] = all;
            }
            __syncthreads();
            before = s_red[0] + s_red[1] + s_red[2] + s_red[3];
            all = s_red[4] + s_red[5] + s_red[6] + s_red[7];
        }
        const bool fits = (long long)le + (long long)all <= (long long)cap;
        if (blockIdx.x == 0 && n0 == 0 && threadIdx.x == 0) {
            lev[level + 2] = fits ? le + (int)all : le;
            if (!fits) atomicMax(&lev[kLevNeed], (int)min((long long)le + all, 0x7fffffffll));
        }
        if (!fits) return;
        // first child of each node of this step
        const int i = n0 + (int)threadIdx.x;
        const bool mine = (int)threadIdx.x < kNodes && i < count;
        const uint32_t nk = mine ? nkids[i] : 0u;
        uint32_t inc = wave_incl_scan_dpp(nk);
        __syncthreads();
        if (lane == 63) s_red[w] = inc;
        __syncthreads();
        for (int k = 0; k < w; ++k) inc += s_red[k];
        const int first = le + (int)(before + inc - nk);
        if (mine) {
            s_off[threadIdx.x] = first;
            wn[lb + i].first = nk ? first : -1;
            wn[lb + i].nchild = (int)nk;
        }
        __syncthreads();
        const int o = threadIdx.x & 7;
        for (int k = 0; k < kNodes && n0 + k < count; k += kThreads / 8) {
            const int j = k + (int)threadIdx.x / 8, ij = n0 + j, node = lb + ij;
            const bool live = ij < count;
            const int kids = live ? (int)nkids[ij] : 0;
            int s = 0, hi = 0;
            if (kids) {
                s = oct_start[(size_t)ij * 8 + o];
                hi = nhi[node];
            }
            int e = __shfl_down(s, 1);
            if (o == 7) e = hi;
            const bool child = kids && e > s;
            const uint32_t m = (uint32_t)(__ballot(child) >> (lane & 56)) & 0xffu;
            if (!child) continue;
            const int r = __popc(m & ((1u << o) - 1u));
            const int c = s_off[j] + r;
            const double sz = size[node];
            const double h = sz * 0.5, q = sz * 0.25;
            nlo[c] = s;
            nhi[c] = e;
            gcx[c] = gcx[node] + ((o & 1) ? q : -q);
            gcy[c] = gcy[node] + ((o & 2) ? q : -q);
            gcz[c] = gcz[node] + ((o & 4) ? q : -q);
            size[c] = h;
            parent[c] = node;
            next[c] = (r < kids - 1) ? c + 1 : next[node];
        }
        __syncthreads();
    }
}

// Levels below the deepest start (and end) at the node count.
__global__ void k_pad_levels(int* __restrict__ lev, int from, int nnodes) {
    const int L = from + (int)threadIdx.x;
    if (L < kLevNeed) lev[L] = nnodes; // (the table's own entries are as they should be)
}

// ---- moments (tree.cc:153-196) + walk-node pack (tree.cc:507-523) --------------------------------
// All leaves in one launch, then the interior nodes level by level from the deepest. The sums
// are added in particle or child order, as the reference's are; only their loads are batched.
struct MomentArgs {
    WNode* wn;
    const int *nlo, *nhi;
    const double *gcx, *gcy, *gcz, *size;
    const double4* src;
    const double* src_soft;
    const uint32_t* orderbuf;
    int* slot_leaf;
    NodeVel nv;
    double *delta_out, *soft_out;
};

// Sums over a node's particles or children.
struct NodeSums {
    double M = 0, sx = 0, sy = 0, sz = 0, smax = 0;
    double vmax = 0, pvx = 0, pvy = 0, pvz = 0; // with velocities: max |v| and momentum
};

__device__ __forceinline__ void put_node(const MomentArgs& a, int node, NodeSums S, int first,
                                         int nk, int lo, int hi) {
    if (S.M > 0) {
        S.sx /= S.M;
        S.sy /= S.M;
        S.sz /= S.M;
    }
    const double dx = S.sx - a.gcx[node], dy = S.sy - a.gcy[node], dz = S.sz - a.gcz[node];
    const double delta = sqrt(dx * dx + dy * dy + dz * dz);
    const double side = a.size[node];
    WNode w;
    w.cx = S.sx;
    w.cy = S.sy;
    w.cz = S.sz;
    w.s = side + delta;
    w.mass = S.M;
    w.soft = (float)S.smax;
    w.len = (float)side;
    w.first = first;
    w.nchild = nk;
    w.plo = lo;
    w.phi = hi;
    a.wn[node] = w;
    a.delta_out[node] = delta;
    a.soft_out[node] = S.smax;
    const NodeVel& nv = a.nv;
    nv.vmax[node] = (float)S.vmax; // 0 without velocities
    if (nv.vx) {
        // centre-of-mass velocity (tree.cc:188-190), the build moments that refreshes start
        // from, and zeroed incremental moments
        const size_t nn = (size_t)nv.nn;
        nv.vcom[node] = (S.M > 0) ? S.pvx / S.M : 0.0;
        nv.vcom[nn + node] = (S.M > 0) ? S.pvy / S.M : 0.0;
        nv.vcom[2 * nn + node] = (S.M > 0) ? S.pvz / S.M : 0.0;
        nv.m0[node] = S.M;
        nv.m0[nn + node] = S.sx;
        nv.m0[2 * nn + node] = S.sy;
        nv.m0[3 * nn + node] = S.sz;
        for (int d = 0; d < 3; ++d) {
            nv.dp[d * nn + node] = 0.0;
            nv.dq[d * nn + node] = 0.0;
        }
        nv.dmass[node] = 0.0;
    }
    nv.xpad[node] = 0.0f;
}

// The leaves, one thread each, four particles loaded together; nleaf (their number) is added to
// once a workgroup (once a wave, it had 18,000 additions in turn at 4M particles).
__global__ __launch_bounds__(kThreads) void k_leaf_moments(int nnodes, MomentArgs a,
                                                           int* __restrict__ nleaf) {
    __shared__ int s_n[kThreads / kWave];
    int mine = 0;
    for (int node = blockIdx.x * kThreads + threadIdx.x; node < nnodes;
         node += gridDim.x * kThreads) {
        if (a.wn[node].nchild != 0) continue;
        ++mine;
        const int lo = a.nlo[node], hi = a.nhi[node];
        NodeSums S;
        for (int k0 = lo; k0 < hi; k0 += 4) {
            double4 p[4];
            double e[4], ux[4], uy[4], uz[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = min(k0 + j, hi - 1);
                p[j] = a.src[k];
                e[j] = a.src_soft[k];
                if (a.nv.vx) {
                    const uint32_t q = a.orderbuf[k];
                    ux[j] = a.nv.vx[q];
                    uy[j] = a.nv.vy[q];
                    uz[j] = a.nv.vz[q];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (k0 + j >= hi) break;
                const double mm = p[j].w;
                S.M += mm;
                S.sx += mm * p[j].x;
                S.sy += mm * p[j].y;
                S.sz += mm * p[j].z;
                if (e[j] > S.smax) S.smax = e[j];
                if (a.nv.vx) { // tree.cc:161-166
                    const double v = sqrt(ux[j] * ux[j] + uy[j] * uy[j] + uz[j] * uz[j]);
                    if (v > S.vmax) S.vmax = v;
                    S.pvx += mm * ux[j];
                    S.pvy += mm * uy[j];
                    S.pvz += mm * uz[j];
                }
                a.slot_leaf[k0 + j] = node;
            }
        }
        put_node(a, node, S, -1, 0, lo, hi);
    }
    for (int d = 32; d >= 1; d >>= 1) mine += __shfl_xor(mine, d);
    if ((threadIdx.x & 63) == 0) s_n[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int n = s_n[0] + s_n[1] + s_n[2] + s_n[3];
        if (n) atomicAdd(nleaf, n);
    }
}

// The interior nodes of one level, one thread each, all children loaded together.
__global__ __launch_bounds__(kThreads) void k_inner_moments(int lb, int count, MomentArgs a) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= count) return;
    const int node = lb + i;
    const int nk = a.wn[node].nchild;
    if (nk == 0) return;
    const int first = a.wn[node].first;
    const NodeVel& nv = a.nv;
    double cm[8], cx[8], cy[8], cz[8], cs[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int c = first + min(j, nk - 1);
        cm[j] = a.wn[c].mass;
        cx[j] = a.wn[c].cx;
        cy[j] = a.wn[c].cy;
        cz[j] = a.wn[c].cz;
        cs[j] = a.soft_out[c];
    }
    NodeSums S;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (j >= nk) break;
        S.M += cm[j];
        S.sx += cm[j] * cx[j];
        S.sy += cm[j] * cy[j];
        S.sz += cm[j] * cz[j];
        if (cs[j] > S.smax) S.smax = cs[j];
    }
    if (nv.vx) { // tree.cc:177-181
        for (int c = first; c < first + nk; ++c) {
            const double mm = a.wn[c].mass;
            if (nv.vmax[c] > S.vmax) S.vmax = nv.vmax[c];
            S.pvx += mm * nv.vcom[c];
            S.pvy += mm * nv.vcom[nv.nn + c];
            S.pvz += mm * nv.vcom[2 * (size_t)nv.nn + c];
        }
    }
    put_node(a, node, S, first, nk, a.nlo[node], a.nhi[node]);
}

// ---- host driver ---------------------------------------------------------------------------------
static gz_status tree_alloc(gz_tree* t, void** p, size_t bytes) {
    *p = nullptr;
    if (t->nblocks == gz_tree::kMaxBlocks)
        return fail(GZ_ERR_INTERNAL, "gz_tree_build: more device blocks than a tree has");
    DevBlock b{};
    GZ_TRY(t->blocks->get(bytes, &b));
    t->block[t->nblocks++] = b;
    *p = b.p;
    return GZ_OK;
}

// Gives a block back while the tree is being built; nothing enqueued may use it any more.
static void tree_drop(gz_tree* t, void* p) {
    for (int i = 0; i < t->nblocks; ++i)
        if (t->block[i].p == p) {
            t->blocks->put(t->block[i]);
            t->block[i] = t->block[--t->nblocks];
            return;
        }
}

template <class T>
static gz_status grow_array(gz_tree* t, T*& a, size_t used, size_t cap, hipStream_t st) {
    void* b = nullptr;
    GZ_TRY(tree_alloc(t, &b, cap * sizeof(T)));
    if (a && used) GZ_HIP(hipMemcpyAsync(b, a, used * sizeof(T), hipMemcpyDeviceToDevice, st));
    if (a) {
        GZ_HIP(hipStreamSynchronize(st));
        tree_drop(t, a);
    }
    a = static_cast<T*>(b);
    return GZ_OK;
}

static gz_status grow_nodes(gz_tree* t, int used, int cap, hipStream_t st) {
    GZ_TRY(grow_array(t, t->wn, used, cap, st));
    GZ_TRY(grow_array(t, t->next, used, cap, st));
    GZ_TRY(grow_array(t, t->parent, used, cap, st));
    GZ_TRY(grow_array(t, t->nlo, used, cap, st));
    GZ_TRY(grow_array(t, t->nhi, used, cap, st));
    GZ_TRY(grow_array(t, t->gcx, used, cap, st));
    GZ_TRY(grow_array(t, t->gcy, used, cap, st));
    GZ_TRY(grow_array(t, t->gcz, used, cap, st));
    GZ_TRY(grow_array(t, t->size, used, cap, st));
    GZ_TRY(grow_array(t, t->delta, used, cap, st));
    GZ_TRY(grow_array(t, t->soft, used, cap, st));
    t->cap = cap;
    return GZ_OK;
}

// The reuse arrays of a tree with nn nodes, in one allocation: vmax and xpad (floats), and with
// velocities vcom (3 nn), the build moments (4 nn: mass, then COM), dp and dq (3 nn each) and
// dmass (nn).
static gz_status alloc_reuse(gz_tree* t, int nn, bool vel) {
    const size_t n = (size_t)std::max(nn, 1);
    const size_t fl = (2 * n * sizeof(float) + 255) & ~size_t(255);
    const size_t db = vel ? 14 * n * sizeof(double) : 0;
    GZ_TRY(tree_alloc(t, &t->reuse_mem, fl + db));
    uint8_t* b = static_cast<uint8_t*>(t->reuse_mem);
    t->vmax = reinterpret_cast<float*>(b);
    t->xpad = t->vmax + n;
    t->has_vel = vel;
    t->vcom = t->m0 = t->dp = t->dq = t->dmass = nullptr;
    if (vel) {
        double* d = reinterpret_cast<double*>(b + fl);
        t->vcom = d;
        t->m0 = d + 3 * n;
        t->dp = d + 7 * n;
        t->dq = d + 10 * n;
        t->dmass = d + 13 * n;
    }
    return GZ_OK;
}

// Work on any stream may still use the blocks (the cache waits for it).
void tree_release(gz_tree* t) {
    t->blocks->retire(t->block, t->nblocks);
    t->nblocks = 0;
    if (t->hmax) (void)hipFree(t->hmax);
}

static float ev_ms(hipEvent_t a, hipEvent_t b) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, a, b) != hipSuccess) return 0.f;
    return ms;
}

gz_status build_tree(gz_ctx* ctx, const gz_particles* p, const gz_build_opts* opts,
                     gz_tree* t) {
    hipStream_t st = ctx->stream;
    const size_t n = p->n;
    if (n >= 0x7FFFFFFFull) return fail(GZ_ERR_INVALID, "gz_tree_build: n=%zu too large", n);
    if (n > 0 && (!p->x || !p->y || !p->z || !p->m))
        return fail(GZ_ERR_INVALID, "gz_tree_build: null position or mass array");
    if (p->zeta) return fail(GZ_ERR_UNSUPPORTED, "gz_tree_build: zeta corrections not supported");
    const long long seed = opts ? opts->randomize_seed : -1;
    const double fx = opts ? opts->shift[0] : 0.0, fy = opts ? opts->shift[1] : 0.0,
                 fz = opts ? opts->shift[2] : 0.0;
    const int max_nodes = opts ? opts->max_nodes : 0;
    const int nc = (opts && opts->n_clusters > 1) ? opts->n_clusters : 1;
    if (nc > 1) {
        if (!opts->cluster_start)
            return fail(GZ_ERR_INVALID, "gz_tree_build: n_clusters > 1 without cluster_start");
        if (seed >= 0 || fx != 0.0 || fy != 0.0 || fz != 0.0)
            return fail(GZ_ERR_UNSUPPORTED, "gz_tree_build: root randomisation with clusters");
        if (opts->cluster_start[0] != 0 || opts->cluster_start[nc] != n)
            return fail(GZ_ERR_INVALID, "gz_tree_build: clusters must cover [0, n)");
        for (int c = 0; c < nc; ++c)
            if (opts->cluster_start[c + 1] < opts->cluster_start[c])
                return fail(GZ_ERR_INVALID, "gz_tree_build: cluster offsets must not decrease");
    }
    t->n = n;
    t->n_clusters = nc;
    hipEvent_t* ev = ctx->ev;
    GZ_HIP(hipEventRecord(ev[0], st));

    // --- bbox + root cell (one per cluster for a forest)
    DevMem& s0 = ctx->scratch[0];
    const unsigned nbb = (unsigned)std::max<size_t>(1, std::min<size_t>(grid_for(n), 1024));
    const size_t s0_live = nbb * 6 * sizeof(double) + 16 * sizeof(double) +
                           (size_t)nc * (4 * sizeof(double) + 2 * sizeof(int)) + 512;
    GZ_TRY(s0.reserve(s0_live + nbb * 4 * sizeof(uint32_t)));
    double* partial = s0.as<double>();
    double* droot = partial + (size_t)nbb * 6;
    double* croots = droot + 16;                                     // nc x 4 (forest)
    int* ccount = reinterpret_cast<int*>(croots + (size_t)4 * nc);   // nc + 1 (forest)
    uint32_t* live = reinterpret_cast<uint32_t*>(s0.as<uint8_t>() + s0_live);
    uint32_t* cstart_dev = nullptr;
    if (nc > 1) {
        GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->cluster_start_dev),
                          (nc + 1) * sizeof(uint32_t)));
        std::vector<uint32_t> hc(nc + 1);
        for (int c = 0; c <= nc; ++c) hc[c] = (uint32_t)opts->cluster_start[c];
        GZ_HIP(hipMemcpy(t->cluster_start_dev, hc.data(), hc.size() * sizeof(uint32_t),
                         hipMemcpyHostToDevice));
        cstart_dev = t->cluster_start_dev;
        k_bbox_clusters<<<nc, kThreads, 0, st>>>(p->x, p->y, p->z, p->m, cstart_dev, croots);
        // droot keeps the first cluster's cell for the tree's info
        GZ_HIP(hipMemcpyAsync(droot, croots, 4 * sizeof(double), hipMemcpyDeviceToDevice, st));
    } else {
        k_bbox_partial<<<nbb, kThreads, 0, st>>>(p->x, p->y, p->z, p->m, n, partial, live);
        k_root_cell<<<1, kThreads, 0, st>>>(partial, live, (int)nbb, seed, fx, fy, fz, droot);
    }
    GZ_HIP(hipGetLastError());
    double hroot[11];
    GZ_HIP(hipMemcpyAsync(hroot, droot, sizeof hroot, hipMemcpyDeviceToHost, st));
    GZ_HIP(hipEventRecord(ev[1], st));

    // --- live filter + keys
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->rank), n * sizeof(uint32_t)));
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->leaf_of), n * sizeof(int)));
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->slot_leaf), n * sizeof(int)));
    const size_t nalloc = std::max<size_t>(n, 1);
    // order / keys ping-pong buffers
    DevMem& s2 = ctx->scratch[2];
    ScratchUse s2_use(s2);
    GZ_TRY(s2.reserve(nalloc * (2 * sizeof(uint64_t) + 2 * sizeof(uint32_t)) + 256));
    uint64_t* k0 = s2.as<uint64_t>();
    uint64_t* k1 = k0 + nalloc;
    uint32_t* v0 = reinterpret_cast<uint32_t*>(k1 + nalloc);
    uint32_t* v1 = v0 + nalloc;
    GZ_HIP(hipStreamSynchronize(st));
    for (int k = 0; k < 4; ++k) t->root_box[k] = hroot[k];
    size_t nl = n;
    // one tree whose particles are all live (the usual case): slot r is particle r before the
    // sort. Otherwise the live ones are compacted first.
    const bool all_live = nc == 1 && hroot[10] == (double)n;
    if (n > 0 && !all_live) {
        DevMem& s1 = ctx->scratch[1];
        const size_t flag_bytes = (nalloc + 64) * sizeof(uint32_t);
        GZ_TRY(s1.reserve(flag_bytes + scan_tmp_bytes(nalloc) + 64));
        uint32_t* flags = s1.as<uint32_t>();
        uint32_t* dcount = flags + nalloc;
        void* stmp = reinterpret_cast<uint8_t*>(s1.p) + flag_bytes;
        k_live_flags<<<grid_for(n), kThreads, 0, st>>>(p->m, n, flags);
        GZ_TRY(exclusive_scan_u32(flags, flags, n, dcount, stmp, st));
        k_live_compact<<<grid_for(n), kThreads, 0, st>>>(p->m, n, flags, v0);
        GZ_HIP(hipGetLastError());
        uint32_t n_live32 = 0;
        GZ_HIP(hipMemcpyAsync(&n_live32, dcount, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        nl = n_live32;
    }
    t->n_live = nl;
    const double* key_roots = nc > 1 ? croots : droot;
    if (nl > 0) {
        k_keys<<<grid_for(nl), kThreads, 0, st>>>(all_live ? nullptr : v0, nl, p->x, p->y, p->z,
                                                  key_roots, cstart_dev, nc, k0, v0);
        GZ_HIP(hipGetLastError());
    }
    GZ_HIP(hipEventRecord(ev[2], st));

    // --- sort (a forest: by key, then stably by cluster, so each cluster is one sorted block)
    GZ_TRY(radix_sort_pairs(k0, v0, k1, v1, nl, 3 * kMaxLevel, ctx->scratch[3], st));
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->skey), nl * sizeof(uint64_t)));
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->orderbuf), nl * sizeof(uint32_t)));
    std::vector<int> rstart_h(nc + 1, 0);
    if (nc > 1 && nl > 0) {
        k_cluster_keys<<<grid_for(nl), kThreads, 0, st>>>(v0, nl, cstart_dev, nc, k1);
        GZ_HIP(hipGetLastError());
        int bits = 1;
        while ((1 << bits) < nc) ++bits;
        GZ_TRY(radix_sort_pairs(k1, v0, k0, v1, nl, bits, ctx->scratch[3], st));
        k_keys<<<grid_for(nl), kThreads, 0, st>>>(v0, nl, p->x, p->y, p->z, key_roots,
                                                  cstart_dev, nc, t->skey, nullptr);
        GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(ccount), nc, st));
        k_cluster_counts<<<grid_for(nl), kThreads, 0, st>>>(v0, nl, cstart_dev, nc, ccount);
        GZ_HIP(hipGetLastError());
        std::vector<int> cnt(nc);
        GZ_HIP(hipMemcpyAsync(cnt.data(), ccount, nc * sizeof(int), hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        for (int c = 0; c < nc; ++c) rstart_h[c + 1] = rstart_h[c] + cnt[c];
    } else if (nl) {
        GZ_HIP(hipMemcpyAsync(t->skey, k0, nl * sizeof(uint64_t), hipMemcpyDeviceToDevice, st));
    }
    if (nl)
        GZ_HIP(hipMemcpyAsync(t->orderbuf, v0, nl * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
    GZ_HIP(hipEventRecord(ev[3], st));

    // --- sorted source copy
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->src), nl * sizeof(double4)));
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->src_soft), nl * sizeof(double)));
    if (n > nl) { // particles outside the tree (the others are written below)
        k_fill_u32<<<grid_for(n), kThreads, 0, st>>>(t->rank, n, 0xFFFFFFFFu);
        k_fill_u32<<<grid_for(n), kThreads, 0, st>>>(reinterpret_cast<uint32_t*>(t->leaf_of), n,
                                                     0xFFFFFFFFu);
        GZ_HIP(hipGetLastError());
    }
    GZ_TRY(gather_sources(p, t->orderbuf, nl, t->src, t->src_soft, ctx->scratch[2], true, st));
    s2.in_use = false;
    GZ_HIP(hipEventRecord(ev[4], st));

    // --- topology, level by level
    int cap = (int)std::min<size_t>((2 * nl) / kLeafMax * 3 + 1024, 0x7FFFFFF0ull);
    if (max_nodes > 0) cap = std::min(cap, max_nodes);
    GZ_TRY(grow_nodes(t, 0, cap, st));
    t->level_begin.clear();
    t->level_begin.push_back(0);
    t->level_begin.push_back(nc);
    t->arena_grows = 0;
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->level_begin_dev), kLevInts * sizeof(int)));
    int* lev = t->level_begin_dev;
    {
        // root: range [0, nl), the root cell, no parent, no successor. An empty particle set
        // still gets a root (a leaf of mass 0), as the reference's build_node does for [0, 0).
        if (nc > 1) {
            // one root per cluster at level 0, each over its block of the sorted order
            int* rstart_d = ccount; // reuse: nc + 1 sorted offsets
            GZ_HIP(hipMemcpyAsync(rstart_d, rstart_h.data(), (nc + 1) * sizeof(int),
                                  hipMemcpyHostToDevice, st));
            if (nc > cap) {
                GZ_TRY(grow_nodes(t, 0, nc + 1024, st));
                cap = nc + 1024;
            }
            k_init_roots<<<grid_for(nc), kThreads, 0, st>>>(nc, croots, rstart_d, t->nlo, t->nhi,
                                                            t->gcx, t->gcy, t->gcz, t->size,
                                                            t->parent, t->next, lev);
            GZ_HIP(hipStreamSynchronize(st)); // rstart_h is a host vector read by the copy
        } else {
            k_init_root<<<1, 1, 0, st>>>(droot, (int)nl, t->nlo, t->nhi, t->gcx, t->gcy, t->gcz,
                                         t->size, t->parent, t->next, lev);
        }
        GZ_HIP(hipGetLastError());
    }
    DevMem& s4 = ctx->scratch[4];
    ScratchUse s4_use(s4);
    // Levels are enqueued in batches, a read-back of the table after each: as many as a tree of nl
    // particles has unless it is deeply clustered, then four at a time.
    int level = 0, batch = 5;
    for (size_t k = nl / (size_t)nc; k > 8; k >>= 3) ++batch;
    for (bool done = false; !done;) {
        // a level holds at most cap nodes; when there is no memory for that many, the next level
        // alone, whose size is known
        auto bytes = [](size_t nodes) {
            return (nodes * 9 + (nodes + kLevelChunk - 1) / kLevelChunk + 1) * sizeof(int) + 768;
        };
        size_t per = (size_t)cap;
        if (!s4.offer(bytes(per))) {
            per = (size_t)(t->level_begin[level + 1] - t->level_begin[level]);
            batch = 1;
            GZ_TRY(s4.reserve(bytes(per)));
        }
        int* oct = s4.as<int>();
        uint32_t* nk = reinterpret_cast<uint32_t*>(oct + 8 * per);
        uint32_t* csum = nk + per;
        const int end = std::min(level + batch, kMaxLevel + 1);
        for (int L = level; L < end; ++L) {
            // nodes of the level: at most 8 children of each node above; and every node but the
            // roots has a parent of more than kLeafMax particles
            long long most = (L < 12) ? ((long long)nc << (3 * L)) : (long long)cap;
            most = std::max<long long>(1, std::min<long long>(most, cap));
            if (L > 0) most = std::min<long long>(most, 8 * ((long long)nl / (kLeafMax + 1)) + 8);
            const unsigned gs = (unsigned)std::min<long long>((most + kLevelChunk - 1) / kLevelChunk,
                                                              4096);
            if (L <= 3)
                k_split<true><<<gs, kThreads, 0, st>>>(L, lev, t->nlo, t->nhi, t->skey, oct, nk,
                                                       csum);
            else
                k_split<false><<<gs, kThreads, 0, st>>>(L, lev, t->nlo, t->nhi, t->skey, oct, nk,
                                                        csum);
            const int chunks = (cap <= kEmitSmall) ? 1 : 4;
            const long long nodes = (long long)chunks * kLevelChunk;
            const unsigned ge = (unsigned)std::min<long long>((most + nodes - 1) / nodes, 1024);
            const bool scan = cap >= kEmitScan;
            if (scan) k_chunk_scan<<<1, 1024, 0, st>>>(L, lev, csum);
            const auto emit = (chunks == 1) ? k_emit<1, false>
                                            : (scan ? k_emit<4, true> : k_emit<4, false>);
            emit<<<ge, kThreads, 0, st>>>(L, cap, lev, nk, csum, oct, t->nlo, t->nhi, t->gcx,
                                          t->gcy, t->gcz, t->size, t->parent, t->next, t->wn);
            GZ_HIP(hipGetLastError());
        }
        int h[kLevInts];
        GZ_HIP(hipMemcpyAsync(h, lev, sizeof h, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        for (; level < end; ++level) {
            if (h[level + 2] > h[level + 1]) {
                t->level_begin.push_back(h[level + 2]);
                continue;
            }
            if (h[kLevNeed] == 0) { // no children: the deepest level (an empty one follows it)
                t->level_begin.push_back(h[level + 1]);
                done = true;
                break;
            }
            // the children of this level outgrew the arena
            const long long need = h[kLevNeed];
            if (need > 0x7FFFFFF0ll)
                return fail(GZ_ERR_NOMEM, "gz_tree_build: node count overflow");
            if (max_nodes > 0)
                return fail(GZ_ERR_ARENA, "gz_tree_build: tree needs more than max_nodes=%d nodes",
                            max_nodes);
            const long long want = std::min<long long>(2 * need + 1024, 0x7FFFFFF0ll);
            GZ_TRY(grow_nodes(t, h[level + 1], (int)want, st));
            cap = (int)want;
            ++t->arena_grows;
            GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(lev + kLevNeed), 1, st));
            break;
        }
        batch = 4;
    }
    s4.in_use = false;
    const int nnodes = t->level_begin.back();
    t->nnodes = nnodes;
    t->depth = (int)t->level_begin.size() - 2;
    // any level index up to kMaxLevel + 1 is valid
    k_pad_levels<<<1, 64, 0, st>>>(lev, (int)t->level_begin.size(), nnodes);
    GZ_HIP(hipGetLastError());
    GZ_HIP(hipEventRecord(ev[5], st));

    // --- reuse state (tree.h:250-317): vmax and xpad always, the velocity moments with velocities
    NodeVel nv{};
    GZ_TRY(alloc_reuse(t, nnodes, opts && opts->vx && opts->vy && opts->vz));
    GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->age), sizeof(double)));
    k_fill_u32<<<1, kThreads, 0, st>>>(reinterpret_cast<uint32_t*>(t->age), 2, 0u);
    nv.nn = nnodes;
    nv.vmax = t->vmax;
    nv.xpad = t->xpad;
    if (t->has_vel) {
        GZ_TRY(tree_alloc(t, reinterpret_cast<void**>(&t->svel),
                      std::max<size_t>(t->n_live, 1) * sizeof(double4)));
        if (t->n_live)
            k_gather_vel<<<grid_for(t->n_live), kThreads, 0, st>>>(t->orderbuf, t->n_live,
                                                                   opts->vx, opts->vy, opts->vz,
                                                                   t->svel);
        GZ_HIP(hipGetLastError());
        nv.vx = opts->vx;
        nv.vy = opts->vy;
        nv.vz = opts->vz;
        nv.vcom = t->vcom;
        nv.m0 = t->m0;
        nv.dp = t->dp;
        nv.dq = t->dq;
        nv.dmass = t->dmass;
    }

    // --- moments + pack, deepest level first
    int* dleaf = reinterpret_cast<int*>(droot + 12);
    k_fill_u32<<<1, kThreads, 0, st>>>(reinterpret_cast<uint32_t*>(dleaf), 1, 0u);
    const MomentArgs ma{t->wn, t->nlo, t->nhi, t->gcx, t->gcy, t->gcz, t->size, t->src,
                        t->src_soft, t->orderbuf, t->slot_leaf, nv, t->delta, t->soft};
    k_leaf_moments<<<std::min(grid_for(nnodes), 4096u), kThreads, 0, st>>>(nnodes, ma, dleaf);
    GZ_HIP(hipGetLastError());
    // (the deepest level is all leaves)
    for (int level = (int)t->level_begin.size() - 4; level >= 0; --level) {
        const int lb = t->level_begin[level], le = t->level_begin[level + 1];
        k_inner_moments<<<grid_for(le - lb), kThreads, 0, st>>>(lb, le - lb, ma);
        GZ_HIP(hipGetLastError());
    }
    if (nl)
        k_particle_links<<<grid_for(nl), kThreads, 0, st>>>(t->orderbuf, t->slot_leaf, nl, t->rank,
                                                            t->leaf_of);
    GZ_HIP(hipGetLastError());
    GZ_HIP(hipEventRecord(ev[6], st));
    int nleaf = 0;
    WNode r;
    GZ_HIP(hipMemcpyAsync(&nleaf, dleaf, sizeof(int), hipMemcpyDeviceToHost, st));
    GZ_HIP(hipMemcpyAsync(&r, t->wn, sizeof r, hipMemcpyDeviceToHost, st));
    GZ_HIP(hipStreamSynchronize(st));
    t->nleaves = nleaf;
    t->root = 0;
    {
        t->root_com[0] = r.cx;
        t->root_com[1] = r.cy;
        t->root_com[2] = r.cz;
        t->root_mass = r.mass;
    }
    t->times.bbox = ev_ms(ev[0], ev[1]);
    t->times.keys = ev_ms(ev[1], ev[2]);
    t->times.sort = ev_ms(ev[2], ev[3]);
    t->times.links = ev_ms(ev[3], ev[4]);
    t->times.recurse = ev_ms(ev[4], ev[5]);
    t->times.pack = ev_ms(ev[5], ev[6]);
    t->times.total = ev_ms(ev[0], ev[6]);
    return GZ_OK;
}

// Refresh the tree's sorted copy of the source particles (positions, masses, softenings) from p,
// for callers that move particles between a build and a walk. The reference walk reads source
// particles from the live arrays (tree.cc:787-788); this library's walk reads the sorted copy.
gz_status regather_sources(gz_ctx* ctx, const gz_particles* p, gz_tree* t) {
    if (p->n != t->n) return fail(GZ_ERR_INVALID, "particle count %zu differs from the tree's %zu",
                                  p->n, t->n);
    // a captured call must not keep the scratch's address, which a later build may replace
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    GZ_HIP(hipStreamIsCapturing(ctx->stream, &cap));
    DevMem none;
    return gather_sources(p, t->orderbuf, t->n_live, t->src, t->src_soft,
                          cap == hipStreamCaptureStatusNone ? ctx->scratch[2] : none, false,
                          ctx->stream);
}

} // namespace gz
