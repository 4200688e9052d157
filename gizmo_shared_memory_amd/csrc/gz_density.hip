// The density / smoothing-length solve of the shared-memory hydro (shmem::density, hydro.h:115-119,
// hydro.cc:150-327), non-periodic and without the neighbour cache or lazy drift.
//
// The reference iterates each target privately: search the tree within h, sum the kernel over the
// gas neighbours, and take a bracket-guarded Newton step on N_eff(h) = ball_vol(h) sum_j W until
// N_eff is within the (widening) tolerance of the neighbour target. Here it is three kernels, each
// adding the reference's terms in the reference's order (its list is in the tree's slot order, which
// is depth first with children in octant order):
//
//   * k_density_round, while many targets are unconverged: every target one step per round, a lane
//     per target and 64 Morton-neighbouring targets per wave. The wave walks the tree once for all
//     of them, up to 64 nodes at a time (their search boxes packed into 32-byte records per call)
//     on a stack kept in depth-first order, stages the particles of the leaves it meets in LDS,
//     and every lane tests each against its own sphere and notes the neighbours' slots in its
//     column of an LDS buffer; whenever some column is nearly full, and at the end, the lanes add
//     their neighbours' terms. The targets that are done leave the active list (a stable
//     compaction, so the waves keep their Morton locality).
//   * k_density_near, for the last kLastTargets: a wave per target, iterated to the end on
//     candidates collected once.
//   * k_density_far, a wave per target on the tree, for spheres that hold many particles: in a
//     round, targets whose radius exceeds kFarLeaf times their leaf's side (one of them would make
//     its wave of 64 walk a large part of the tree), and among the last, those with more than
//     kNearMax candidates, or all when that many neighbours are wanted.
//
// What bounds a round: at 4.2M targets (Hernquist, 3% from converged) 38,500 VALU instructions a
// wave, busy 4.4 of 7.0 ms, the rest latency at 2.5 waves per SIMD (LDS): about 14 instructions for
// each of some 1,000 staged particles, and 81 steps of about 110 for the terms (33 neighbours a
// lane; a buffer fills with the lanes unevenly advanced). Walking one node at a time with the
// general square root and division it took 8.9 ms. The neighbours' live values are put in slot
// order once per call, where a wave's lanes find them in the same lines.
//
// The one difference from the reference's arithmetic is pow(dx, 2) in the 3D face-closure test,
// taken here as dx * dx (correctly rounded; glibc's pow is within half an ulp of it, not always
// equal).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "gz_features.h"
#include "gz_internal.h"
#include "gz_spheres.h"
#include "gz_wave.h"

namespace gz {
namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr int kMaxIter = 100; // hydro.cc:201
constexpr int kNbBuf = 32;          // neighbours each lane holds before their terms are added
constexpr double kFarLeaf = 4.0;    // radius over leaf side beyond which a target takes a wave
// The last active targets iterate to the end in one launch. Rounds are cheaper per target while a
// wave's targets are neighbours; the fewer are left, the further apart they lie and the more
// launches and read-backs they cost. How many are the last, and which kernel takes them, depends on
// how well a converged target's candidates (wanted neighbours times the volume of kNearMargin) fit
// the 256 that k_density_near holds. ms a solve, guesses 2% off, by the limit and the kernel:
//
//   neighbours (candidates)      32 (49)   64 (97)   128 (195)  150 (228)  200 (304)  300 (456)
//   300k Hernquist, 131,072 near    2.26      2.22      3.60       4.08       5.51       8.50
//                   393,216 near    2.40      2.37      4.00       6.21      16.0       24.3
//                   131,072 far     4.27      2.39      3.60       4.09       5.29       7.86
//   300k halo+disk, 131,072 near    2.72      3.27      5.80       6.80       9.56      13.9
//                   393,216 near    2.65      2.79      5.08       7.17      15.4       24.3
//                   131,072 far     5.25      3.28      5.84       6.90       9.11      13.3
//   60k Hernquist,  131,072 near     .73       .71      1.15       1.71       3.71       5.35
//                   131,072 far     2.71      1.54      2.46       2.74       3.34       4.63
//   1M Hernquist,   131,072 near    7.19      5.68      9.34      10.7       13.6       20.5
//                   393,216 near    7.17      5.69      9.39      10.7       13.6       23.3
//                   131,072 far     8.42      5.78      9.77      11.3       14.8       20.5
//   4.2M Hernquist, 131,072 near   23.0                35.5                  53.5       73.2
//                   393,216 near   22.6                35.5                  51.0       73.2
//
// So near to 310 candidates, of which up to 393,216 targets to 200 candidates, else 131,072.
constexpr uint32_t kLastTargets = 393216, kLastTargetsFull = 131072;
constexpr double kCollectMost = 200.0, kCollectMax = 310.0;
// Up to this many targets the launch's time is its slowest target's, and one that starts from a
// radius far too large takes that long twice in two kernels: 1,000 targets of 1M from rough guesses
// .83 ms in two, .52 in one; from good ones .43 and .45, and 6% more for 8,000.
constexpr uint32_t kNearFar = 2048;

// kernel_norm, ball_vol, kernel_w, kernel_dwdh (hydro.h:29-65): cubic spline of support h in dim
// dimensions, operand for operand.
__device__ __forceinline__ double knorm(double h, int dim) {
    if (dim == 1) return (4.0 / 3.0) / h;
    if (dim == 2) return 40.0 / (7.0 * kPi * h * h);
    return 8.0 / (kPi * h * h * h);
}
__device__ __forceinline__ double ball_vol(double h, int dim) {
    if (dim == 1) return 2.0 * h;
    if (dim == 2) return kPi * h * h;
    return 4.0 * kPi / 3.0 * h * h * h;
}
// The correctly rounded square root and quotient, as the IEEE operations give them, in fewer
// instructions than the compiler's general expansions (which scale for the whole exponent range):
// the hardware's estimate or a rounded reciprocal, refined with fused multiply-adds until the last
// correction is a rounding of the exact remainder (P. Markstein, IBM J. Res. Dev. 34 (1990) 111).
// Outside the ranges where every intermediate is exact the general operation is used.
// most: a bound on the root, applied only outside the range.
__device__ __forceinline__ double sqrt_rn(double x, double most) {
    if ((x > 0.0 && x < 1e-250) || !(x <= 1e250)) {
        const double r = sqrt(x);
        return r > most ? most : r;
    }
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return (x > 0.0) ? g : x; // (0 stays 0)
}

// W(r) and dW/dh(r) (hydro.h:36-65) for one support h: operand for operand, with what depends on
// h alone computed once.
struct Kernel {
    double h, rh, norm, norm2, c1; // rh = 1/h; norm2 = norm * 2; c1 = -(dim / h) * norm
    bool general;                  // h outside the range of the short quotient
    __device__ __forceinline__ void set(double h_, int dim) {
        h = h_;
        rh = 1.0 / h;
        norm = knorm(h, dim);
        norm2 = norm * 2.0;
        c1 = -((double)dim / h) * norm;
        general = !(h > 1e-120 && h < 1e120);
    }
    // The distance of a square. Where the short quotient serves, distances end at 1e187, far outside
    // any kernel: the quotient of a larger one (a particle that has moved to infinity since the
    // tree took its position) could be infinite, and its correction NaN.
    __device__ __forceinline__ double distance(double x) const {
        return sqrt_rn(x, general ? __builtin_inf() : 1e187);
    }
    // a / h (a of a size where a quotient that underflows changes no sum it enters)
    __device__ __forceinline__ double over_h(double a) const {
        if (general) return a / h;
        double q = a * rh;
        q = __builtin_fma(__builtin_fma(-q, h, a), rh, q);
        return __builtin_fma(__builtin_fma(-q, h, a), rh, q);
    }
    __device__ __forceinline__ void at(double r, double* w, double* dwdh) const {
        const double q = over_h(r);
        const double t = 6.0 * q * q, u = 1.0 - q;
        const double f_in = 1.0 - t + t * q, f_out = 2.0 * u * u * u;
        const double fp_in = -12.0 * q + 18.0 * q * q, fp_out = -6.0 * u * u;
        const bool in = q < 0.5;
        const double f = in ? f_in : f_out, fp = in ? fp_in : fp_out;
        const double ww = in ? norm * f_in : norm2 * u * u * u;
        const double d = c1 * f - over_h(q) * norm * fp;
        *w = (q >= 1.0) ? 0.0 : ww;
        *dwdh = (q >= 1.0) ? 0.0 : d;
    }
};

// invert_moments (shmem/vec.h:43-63) of the symmetric moments e (xx yy zz xy yz xz) into b
// (row-major 3x3, zero outside the live block); false when degenerate. 3D is Mat3::invert
// (math_types/mat3.h:41-67): cofactors times 1 / det, singular when det is 0 or NaN.
__device__ __forceinline__ bool invert_moments(const double* e, double* b, int dim) {
#pragma unroll
    for (int k = 0; k < 9; ++k) b[k] = 0.0;
    if (dim == 1) {
        if (fabs(e[0]) < 1e-300) return false;
        b[0] = 1.0 / e[0];
        return true;
    }
    if (dim == 2) {
        const double det = e[0] * e[1] - e[3] * e[3];
        if (fabs(det) < 1e-300) return false;
        b[0] = e[1] / det;
        b[1] = -e[3] / det;
        b[3] = -e[3] / det;
        b[4] = e[0] / det;
        return true;
    }
    const double m00 = e[0], m01 = e[3], m02 = e[5], m10 = e[3], m11 = e[1], m12 = e[4],
                 m20 = e[5], m21 = e[4], m22 = e[2];
    const double d = m00 * (m11 * m22 - m12 * m21) - m01 * (m10 * m22 - m12 * m20) +
                     m02 * (m10 * m21 - m11 * m20);
    if (d == 0.0 || d != d) return false;
    const double id = 1.0 / d;
    b[0] = (m11 * m22 - m12 * m21) * id;
    b[1] = (m02 * m21 - m01 * m22) * id;
    b[2] = (m01 * m12 - m02 * m11) * id;
    b[3] = (m12 * m20 - m10 * m22) * id;
    b[4] = (m00 * m22 - m02 * m20) * id;
    b[5] = (m02 * m10 - m00 * m12) * id;
    b[6] = (m10 * m21 - m11 * m20) * id;
    b[7] = (m01 * m20 - m00 * m21) * id;
    b[8] = (m00 * m11 - m01 * m10) * id;
    return true;
}

// A read of memory no kernel of the solve writes (the tree's records), through the constant
// address space: at a wave-uniform address it is a scalar load, served by the scalar cache.
template <class T>
__device__ __forceinline__ T ld_const(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "read as whole dwords");
    const __attribute__((address_space(4))) uint32_t* q =
        (const __attribute__((address_space(4))) uint32_t*)p;
    uint32_t w[sizeof(T) / 4];
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i) w[i] = q[i];
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

struct DensArgs {
    const uint32_t* act; // active targets (positions in the target list), in slot order
    int n_act;
    const uint32_t* targets;
    const double *x, *y, *z, *m;
    const uint8_t* type; // null: all gas
    // the particles' live values by slot (x, y, z, m, and whether gas), or null: read through
    // orderbuf from the arrays above
    const double4* live;
    const uint8_t* live_gas;
    double des_ngb, ngb_tol;
    int n_dims;
    const double* cond_prev; // by particle, or null
    double *h, *h_lo, *h_hi, *rho;
    int *iter, *nngb, *iters;
    uint32_t* keep; // 1: the target stays active
    // the rounds: a target whose radius exceeds kFarLeaf times its leaf's side is left to a wave
    // of its own (appended to far_list)
    const int* tslot;     // sorted slot per target (list position), -1 outside the tree
    const int* slot_leaf;
    uint32_t* far_list;
    uint32_t* n_far;
    // the tree: its search nodes (built per call), the side of each node (the far test), the
    // sorted copy of the particles and their indices, the roots, and the time since the build
    // (the vmax pad)
    SphereNodes nodes;
    const WNode* wn;
    const double* size;
    const double4* src;
    const uint32_t* orderbuf;
};

// The terms one gas neighbour j adds to a target at (p0, p1, p2) with support h (hydro.cc:206-217):
// v = {W, dW/dh, m W, dx dx W, dy dy W, dz dz W, dx dy W, dy dz W, dx dz W, dx W, dy W, dz W}, and
// whether r < h. Non-gas neighbours add nothing (returns false).
constexpr int kTerms = 12;
__device__ __forceinline__ int wave_max_i(int v) {
    for (int d = 32; d >= 1; d >>= 1) v = max(v, __shfl_xor(v, d));
    return v;
}
struct Neighbour {
    double x, y, z, m;
    bool gas;
};
__device__ __forceinline__ Neighbour neighbour_at(const DensArgs& a, uint32_t slot) {
    Neighbour n;
    if (a.live) {
        const double4 q = a.live[slot];
        n.x = q.x; n.y = q.y; n.z = q.z; n.m = q.w;
        n.gas = !a.live_gas || a.live_gas[slot] != 0;
    } else {
        const uint32_t j = a.orderbuf[slot];
        n.x = a.x[j]; n.y = a.y[j]; n.z = a.z[j]; n.m = a.m[j];
        n.gas = !a.type || a.type[j] == 0;
    }
    return n;
}
__device__ __forceinline__ bool density_terms(const Neighbour& nb, double p0, double p1, double p2,
                                              const Kernel& kern, double* v, bool* inside) {
    if (!nb.gas) return false; // gas neighbours only
    const double d0 = nb.x - p0, d1 = nb.y - p1, d2 = nb.z - p2;
    const double r = kern.distance(d0 * d0 + d1 * d1 + d2 * d2);
    double w;
    kern.at(r, &w, &v[1]);
    v[0] = w;
    v[2] = nb.m * w;
    v[3] = d0 * d0 * w;
    v[4] = d1 * d1 * w;
    v[5] = d2 * d2 * w;
    v[6] = d0 * d1 * w;
    v[7] = d1 * d2 * w;
    v[8] = d0 * d2 * w;
    v[9] = d0 * w;
    v[10] = d1 * w;
    v[11] = d2 * w;
    *inside = r < kern.h;
    return true;
}

// A target's sums over its neighbours, added in list (traversal) order.
struct DensSums {
    double s[kTerms];
    int n_inside;
};

// A target's solve between steps: its radius, the bracket, the iteration.
struct DensState {
    double h, lo, hi;
    int it;
};

// The rest of one step (hydro.cc:218-296) from the target's sums: the final pass's outputs when
// out of iterations, else the corrections, the convergence test and the Newton / bisection step.
// True: the target is done (its outputs written by a lane with `write`, its radius is st.h).
__device__ bool density_step(const DensArgs& a, uint32_t t, uint32_t p, DensState& st,
                             const DensSums& S, bool write) {
    const int dim = a.n_dims;
    const double h = st.h;
    const int it = st.it;
    if (it >= kMaxIter) {
        // out of iterations: rho and the count at the last h (hydro.cc:285-295)
        if (write) {
            a.rho[t] = S.s[2];
            a.nngb[t] = S.n_inside;
            a.iters[t] = kMaxIter;
        }
        return true;
    }
    const double weight_sum = S.s[0], dweight_dh = S.s[1];
    const double* mom = S.s + 3;
    const double* face = S.s + 9;
    const double n_eff = ball_vol(h, dim) * weight_sum;
    // the condition-number and face-closure corrections widen the neighbour target
    // (hydro.cc:220-262)
    double ncorr = 1.0;
    if (a.cond_prev) {
        const double cn = a.cond_prev[p];
        if (cn > 100.0) ncorr = fmin(sqrt(1.0 + (cn - 100.0) / 1000.0), 2.0);
    }
    double des_eff = a.des_ngb * ncorr, tol_eff = a.ngb_tol * ncorr;
    if (weight_sum > 0) {
        double bm[9];
        if (invert_moments(mom, bm, dim)) {
            const double vol = 1.0 / weight_sum;
            const double dx_i = sqrt(vol * (mom[0] + mom[1] + mom[2]));
            double sum_abs = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double lk =
                    (bm[3 * c] * face[0] + bm[3 * c + 1] * face[1] + bm[3 * c + 2] * face[2]) *
                    (2.0 * vol);
                sum_abs += fabs(lk) / dim;
            }
            const double pw = (dim == 3) ? dx_i * dx_i : (dim == 2 ? dx_i : 1.0);
            const double denom = 2.0 * dim * pw;
            if (denom > 0) {
                const double fce = sum_abs / denom;
                if (fce > 0.35) ncorr = fmax(ncorr, fmin(fce / 0.35, 2.0));
                des_eff = a.des_ngb * ncorr;
                tol_eff = a.ngb_tol * ncorr;
            }
        }
    }
    // the tolerance widens as the solve iterates (hydro.cc:263-267)
    if (it > 1)
        tol_eff = fmin(0.25 * des_eff, tol_eff * exp(0.1 * log(des_eff / (16.0 * tol_eff)) * it));
    const double residual = n_eff - des_eff;
    if (fabs(residual) < tol_eff) {
        if (write) {
            a.rho[t] = S.s[2];
            a.nngb[t] = S.n_inside;
            a.iters[t] = it;
        }
        return true;
    }
    double h_lo = st.lo, h_hi = st.hi;
    if (residual > 0) h_hi = h;
    else h_lo = h;
    // Newton on N_eff(h), guarded by the bracket (hydro.cc:271-281)
    const double dneff_dh = ball_vol(h, dim) * ((double)dim / h * weight_sum + dweight_dh);
    double h_next = (dneff_dh > 0) ? h - residual / dneff_dh : 0.0;
    if (h_next <= h_lo || (h_hi > 0 && h_next >= h_hi) || h_next <= 0) {
        if (h_hi > 0) h_next = (h_lo > 0) ? sqrt(h_lo * h_hi) : 0.5 * h_hi;
        else h_next = h * ((residual > 0) ? 0.7 : 1.6);
    }
    st = {h_next, h_lo, h_hi, it + 1};
    return false;
}

// A step whose state lives in memory; keep: the target (entry k of the active list) goes on.
__device__ void density_update(const DensArgs& a, int k, uint32_t t, uint32_t p, double h, int it,
                               const DensSums& S) {
    DensState st{h, a.h_lo[t], a.h_hi[t], it};
    if (density_step(a, t, p, st, S, true)) {
        a.keep[k] = 0;
        return;
    }
    a.h[t] = st.h;
    a.h_lo[t] = st.lo;
    a.h_hi[t] = st.hi;
    a.iter[t] = st.it;
    a.keep[k] = 1;
}

// Packed sums: the neighbours' terms lie in s_v in traversal order, and lane c < 12 adds term c of
// each to acc. Eight are read together: the additions stay in order, their reads do not wait for
// each other.
__device__ __forceinline__ double add_terms(const double (*s_v)[65], int lane, int n, double acc) {
    if (lane < kTerms) {
        const double* v = s_v[lane];
        int i = 0;
        for (; i + 8 <= n; i += 8) {
            double u[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) u[j] = v[i + j];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc += u[j];
        }
        for (; i < n; ++i) acc += v[i];
    }
    return acc;
}

// A step's sums for one target by a whole wave on the tree, the search walked depth first. The lanes
// test a node's children together (a forest's roots up to 64 at a time), so the wave takes one step
// per admitted interior node; the admitted leaves among a node's children up to its next admitted
// interior child are taken together, their particles (contiguous slot ranges) spread over the
// lanes in slot order, tested against the sphere, and the neighbours' terms computed into s_v in
// that order. Lane c (c < 12) then adds term c of each, in order, so every sum is the round's, term
// by term.
__device__ __forceinline__ void far_sums(const DensArgs& a, double qx, double qy, double qz, double h,
                                         double (*s_v)[65], DensSums* out) {
    const int lane = threadIdx.x;
    const int r_first = (a.nodes.nclusters > 1) ? 0 : a.nodes.root;
    const int r_count = (a.nodes.nclusters > 1) ? a.nodes.nclusters : 1;
    const double r2 = h * h; // the search's radius_sq (hydro.cc:50)
    Kernel kern;
    kern.set(h, a.n_dims);
    // the node test of the forward search (hydro.cc:55-72), as the rounds evaluate it
    auto admits = [&](const SRec& nr) -> bool {
        double dist = h + (double)nr.half + (double)nr.xpad;
        if (a.nodes.tau > 0) dist += (double)nr.vmax * a.nodes.tau;
        const double dx = (double)nr.cx - qx, dy = (double)nr.cy - qy,
                     dz = (double)nr.cz - qz;
        if ((dx > dist || -dx > dist) || (dy > dist || -dy > dist) ||
            (dz > dist || -dz > dist))
            return false;
        const double ds = dist + 0.7320508075688772 * (double)nr.half;
        return !(dx * dx + dy * dy + dz * dz > ds * ds);
    };
    double acc = 0.0; // lane c < 12: term c's sum
    int n_in = 0;     // the count inside h (the same in every lane)
    int nbuf = 0;     // neighbours waiting in s_v (the same in every lane)
    auto flush = [&]() {
        __syncthreads();
        acc = add_terms(s_v, lane, nbuf, acc);
        __syncthreads();
        nbuf = 0;
    };
    // one particle per lane (slot s, or none for s < 0): a neighbour when within the radius
    // (the tree's copy of the position, as the search tests it), its terms packed into s_v
    // in lane order
    auto take = [&](int s) {
        double v[kTerms];
        bool inside = false, ok = false;
        if (s >= 0) {
            const double4 q = a.src[s];
            const double ex = q.x - qx, ey = q.y - qy, ez = q.z - qz;
            if (ex * ex + ey * ey + ez * ez < r2)
                ok = density_terms(neighbour_at(a, s), qx, qy, qz, kern, v, &inside);
        }
        const uint64_t om = __ballot(ok);
        if (om == 0) return;
        const int n_ok = __builtin_popcountll(om);
        if (nbuf + n_ok > 64) flush();
        if (ok) {
            const int pos = nbuf + lanes_under(om);
#pragma unroll
            for (int c = 0; c < kTerms; ++c) s_v[c][pos] = v[c];
        }
        n_in += __builtin_popcountll(__ballot(ok && inside));
        nbuf += n_ok;
    };
    // the admitted leaves run (bit j: child cf + j), their particles in slot order
    auto leaves = [&](int cf, uint64_t run) {
        int plo = 0, cnt = 0, off = 0, total = 0;
        if ((run >> lane) & 1ull) {
            const SRec c = a.nodes.srec[cf + lane];
            plo = ~c.link;
            cnt = c.span - plo;
        }
        for (uint64_t r = run; r != 0; r &= r - 1) {
            const int j = (int)__builtin_ctzll(r);
            if (lane == j) off = total;
            total += __builtin_amdgcn_readlane(cnt, j);
        }
        for (int g0 = 0; g0 < total; g0 += 64) {
            const int g = g0 + lane;
            int s = -1;
            for (uint64_t r = run; r != 0; r &= r - 1) {
                const int j = (int)__builtin_ctzll(r);
                const int o = __builtin_amdgcn_readlane(off, j);
                if (g >= o && g < o + __builtin_amdgcn_readlane(cnt, j))
                    s = __builtin_amdgcn_readlane(plo, j) + (g - o);
            }
            take(s);
        }
    };
    // A node whose box (its centre and half side as the node test reads them, so the cells
    // below it too) lies inside the sphere, by a margin above the float rounding of node
    // centres: every node below it is admitted, so the walk would test each of its particles
    // in slot order. They are a contiguous slot range, taken 64 at a time instead.
    auto inside_sphere = [&](const SRec& nr) -> bool {
        const double hf = (double)nr.half;
        const double ax = fabs((double)nr.cx - qx) + hf, ay = fabs((double)nr.cy - qy) + hf,
                     az = fabs((double)nr.cz - qz) + hf;
        const double m = 1e-6 * (fabs((double)nr.cx) + fabs((double)nr.cy) +
                                 fabs((double)nr.cz));
        const double hm = h * (1.0 - 1e-12) - m;
        return hm > 0 && ax * ax + ay * ay + az * az < hm * hm;
    };
    for (int r0 = 0; r0 < r_count; r0 += 64) {
        // the children of the node being walked (first index; lane masks of those admitted
        // and not yet visited, and of those that are leaves) and the stack of the same above
        // it, entry d in lane d
        int cf = r_first + r0;
        uint64_t cm, lm;
        {
            bool hit = false, leaf = false;
            if (lane < min(64, r_count - r0)) {
                const SRec c = a.nodes.srec[cf + lane];
                hit = admits(c);
                leaf = c.link < 0;
            }
            cm = __ballot(hit);
            lm = __ballot(hit && leaf);
        }
        int sp = 0, stf = 0, sml = 0, smh = 0, sll = 0, slh = 0;
        for (;;) {
            if (cm == 0) {
                if (sp == 0) break;
                --sp;
                cf = __builtin_amdgcn_readlane(stf, sp);
                cm = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(smh, sp) << 32) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readlane(sml, sp);
                lm = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(slh, sp) << 32) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readlane(sll, sp);
                continue;
            }
            const uint64_t inner = cm & ~lm;
            if ((cm & (0 - cm) & lm) != 0) {
                // the next child is a leaf: it and the leaves after it up to the next
                // interior child
                const uint64_t run = inner ? (cm & ((inner & (0 - inner)) - 1)) : cm;
                cm &= ~run;
                leaves(cf, run);
                continue;
            }
            // an interior child: its admitted children are walked before its remaining
            // siblings, which wait on the stack
            const int node = cf + (int)__builtin_ctzll(cm);
            cm &= cm - 1;
            const SRec nr = ld_const(a.nodes.srec + node);
            if (inside_sphere(nr)) {
                const WNode w = ld_const(a.wn + node);
                for (int s0 = w.plo; s0 < w.phi; s0 += 64)
                    take(s0 + lane < w.phi ? s0 + lane : -1);
                continue;
            }
            bool hit = false, leaf = false;
            if (lane < nr.span) {
                const SRec c = a.nodes.srec[nr.link + lane];
                hit = admits(c);
                leaf = c.link < 0;
            }
            const uint64_t om = __ballot(hit);
            if (om == 0) continue;
            if (cm != 0) {
                const bool top = lane == sp;
                stf = top ? cf : stf;
                sml = top ? (int)(uint32_t)cm : sml;
                smh = top ? (int)(uint32_t)(cm >> 32) : smh;
                sll = top ? (int)(uint32_t)lm : sll;
                slh = top ? (int)(uint32_t)(lm >> 32) : slh;
                ++sp;
            }
            cf = nr.link;
            cm = om;
            lm = __ballot(hit && leaf);
        }
    }
    flush();
#pragma unroll
    for (int c = 0; c < kTerms; ++c) out->s[c] = __shfl(acc, c);
    out->n_inside = n_in;
}

// Targets whose spheres reach far beyond their leaf, a wave each (a.act[e] for block e): one step, or
// with LOOP their steps to the end.
template <bool LOOP>
__global__ __launch_bounds__(64) void k_density_far(DensArgs a) {
    __shared__ double s_v[kTerms][65]; // rows padded so the 12 adding lanes hit distinct banks
    const int e = blockIdx.x;
    const uint32_t t = a.act[e];
    const uint32_t p = a.targets[t];
    const double qx = a.x[p], qy = a.y[p], qz = a.z[p];
    for (;;) {
        const double h = a.h[t];
        const int it = a.iter[t];
        DensSums S;
        far_sums(a, qx, qy, qz, h, s_v, &S);
        if (threadIdx.x == 0) density_update(a, e, t, p, h, it, S);
        if (!LOOP) break;
        __syncthreads(); // the update's state, written by lane 0, for every lane
        if (a.keep[e] == 0) break;
    }
}

// The last targets, a wavefront each (target a.act[e] for block e), iterated to the end. The wave
// collects its target's candidates once, out to kNearMargin times the radius, up to 64 nodes in
// depth-first order at a time, and keeps them in registers (candidate 64 k + lane), in slot order: a
// step is then a distance test and the terms of those inside, without the tree, until the radius
// outgrows the collection (one of a radius above zero). (Targets that run to the 100-iteration cap,
// whose walks one node at a time set the launch's time, took 39 us a step before, and 2-3 us now.)
// When some particle has left its cell the candidates are collected for each step at its own radius,
// under the reference's node tests.
//
// A sphere of more than kNearMax candidates is left to k_density_far (appended to far_list, its state
// in memory), or with FAR takes its steps from far_sums here until it has shrunk: a launch less, but
// more registers. Whether it will be one is then told in advance, since a collection that overflows
// is thrown away: at first by the leaf's side, as in the rounds, then from the step before, whose
// neighbours fill the next sphere in proportion to its volume.
constexpr int kNearSlots = 4; // candidates a lane holds
constexpr int kNearMax = 64 * kNearSlots;
constexpr double kNearMargin = 1.15;
// The volume out to which candidates are collected for a sphere of g times the radius, over this one's.
__host__ __device__ __forceinline__ double near_volume(double g, int dim) {
    g *= kNearMargin;
    return (dim == 3) ? g * g * g : (dim == 2 ? g * g : g);
}
template <bool FAR>
__global__ __launch_bounds__(64, 3) void k_density_near(DensArgs a) {
    // the collection's stack and leaf runs, then a step's packed terms
    __shared__ union {
        double v[kTerms][65]; // rows padded so the 12 adding lanes hit distinct banks
        struct {
            int stk[kSphStack], lpre[64], lplo[64];
        } w;
    } s;
    __shared__ uint32_t s_cand[kNearMax];
    const int lane = threadIdx.x;
    const int e = blockIdx.x;
    const uint32_t t = a.act[e];
    const uint32_t p = a.targets[t];
    const double qx = a.x[p], qy = a.y[p], qz = a.z[p];
    const bool fresh = *a.nodes.moved == 0;
    DensState st{a.h[t], a.h_lo[t], a.h_hi[t], a.iter[t]};
    double cx[kNearSlots], cy[kNearSlots], cz[kNearSlots]; // the tree's copy of the positions
    Neighbour nb[kNearSlots];
    int nc = 0;
    double hc = 0.0;   // the radius the candidates reach
    bool have = false; // they can serve another step
    bool full = false; // FAR: this step by far_sums
    if (FAR) {
        const int ts = a.tslot[t];
        full = ts >= 0 && st.h > kFarLeaf * a.size[a.slot_leaf[ts]];
    }

    for (;;) {
        if (!full && !(have && st.h <= hc)) {
            // collect: the search at radius hc, its particles tested against the sphere
            hc = (fresh && st.h > 0) ? st.h * kNearMargin : st.h;
            const double c2 = hc * hc;
            nc = 0;
            walk_sphere<true>(a.nodes, qx, qy, qz, hc, s.w.stk, s.w.lpre, s.w.lplo,
                              [&](bool some, int slot, const double4& q) {
                const double ex = q.x - qx, ey = q.y - qy, ez = q.z - qz;
                const bool in = some && ex * ex + ey * ey + ez * ez < c2;
                const uint64_t im = __ballot(in);
                const int pos = nc + lanes_under(im);
                if (in && pos < kNearMax) s_cand[pos] = (uint32_t)slot;
                nc += __builtin_popcountll(im);
                return nc <= kNearMax;
            });
            if (!FAR && nc > kNearMax) {
                if (lane == 0) {
                    a.h[t] = st.h;
                    a.h_lo[t] = st.lo;
                    a.h_hi[t] = st.hi;
                    a.iter[t] = st.it;
                    a.far_list[atomicAdd(a.n_far, 1u)] = (uint32_t)e;
                }
                return;
            }
            full = nc > kNearMax;
            have = fresh && st.h > 0; // (a negative radius's next step may be larger in size)
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kNearSlots; ++k) {
                if (FAR) {
                    cx[k] = cy[k] = cz[k] = 0.0;
                    nb[k] = Neighbour{};
                }
                if (!full && 64 * k + lane < nc) {
                    const uint32_t slot = s_cand[64 * k + lane];
                    const double4 q = a.src[slot];
                    cx[k] = q.x; cy[k] = q.y; cz[k] = q.z;
                    nb[k] = neighbour_at(a, slot);
                }
            }
        }
        DensSums S;
        if (FAR && full) {
            have = false;
            far_sums(a, qx, qy, qz, st.h, s.v, &S);
#pragma unroll
            for (int k = 0; k < kNearSlots; ++k) { // (held in no register while far_sums runs)
                cx[k] = cy[k] = cz[k] = 0.0;
                nb[k] = Neighbour{};
            }
        } else {
            const double r2 = st.h * st.h;
            Kernel kern;
            kern.set(st.h, a.n_dims);
            double acc = 0.0;
            int n_in = 0, nbuf = 0;
#pragma unroll
            for (int k = 0; k < kNearSlots; ++k) {
                if (64 * k >= nc) break;
                double v[kTerms];
                bool inside = false, ok = false;
                if (64 * k + lane < nc) {
                    const double ex = cx[k] - qx, ey = cy[k] - qy, ez = cz[k] - qz;
                    if (ex * ex + ey * ey + ez * ez < r2)
                        ok = density_terms(nb[k], qx, qy, qz, kern, v, &inside);
                }
                const uint64_t om = __ballot(ok);
                const int n_ok = __builtin_popcountll(om);
                if (nbuf + n_ok > 64) {
                    __syncthreads();
                    acc = add_terms(s.v, lane, nbuf, acc);
                    nbuf = 0;
                }
                __syncthreads();
                if (ok) {
                    const int pos = nbuf + lanes_under(om);
#pragma unroll
                    for (int c = 0; c < kTerms; ++c) s.v[c][pos] = v[c];
                }
                n_in += __builtin_popcountll(__ballot(ok && inside));
                nbuf += n_ok;
            }
            __syncthreads();
            acc = add_terms(s.v, lane, nbuf, acc);
            __syncthreads();
#pragma unroll
            for (int c = 0; c < kTerms; ++c) S.s[c] = __shfl(acc, c);
            S.n_inside = n_in;
        }
        const double h = st.h;
        if (density_step(a, t, p, st, S, lane == 0)) break;
        if (FAR) full = S.n_inside * near_volume(st.h / h, a.n_dims) > (double)kNearMax;
    }
    if (lane == 0) a.h[t] = st.h;
}

// One step for every active target (see the top of the file): lane l of wave w holds active entry
// 64 w + l. A target whose radius reaches far beyond its own leaf would
// make its wave walk a large part of the tree one node at a time; it is queued for a wave of its
// own (k_density_far) and takes no part here.
__global__ __launch_bounds__(64, 3) void k_density_round(DensArgs a) {
    const int lane = threadIdx.x;
    // Block b runs on XCD b % 8: each XCD gets one contiguous share of the Morton-ordered waves.
    const int b = blockIdx.x, nb = gridDim.x;
    const int xcd = b & 7, per = nb >> 3, rem = nb & 7;
    const int wv = xcd * per + min(xcd, rem) + (b >> 3);
    const int k = wv * 64 + lane;
    const bool live = k < a.n_act;
    const int dim = a.n_dims;
    uint32_t t = 0, p = 0;
    double qx = 0, qy = 0, qz = 0, h = 0;
    int it = 0;
    bool mine = false; // this lane steps its target here
    bool far = false;  // this lane's target is left to a wave of its own
    if (live) {
        t = a.act[k];
        p = a.targets[t];
        qx = a.x[p];
        qy = a.y[p];
        qz = a.z[p];
        h = a.h[t];
        it = a.iter[t];
        mine = true;
        const int ts = a.tslot[t];
        if (ts >= 0 && h > kFarLeaf * a.size[a.slot_leaf[ts]]) {
            far = true;
            mine = false;
        }
    }
    // Each lane's neighbours (slots, in traversal order) wait in its column of s_nb until some
    // column is full or the walk ends; then every lane adds its waiting neighbours' terms, in
    // order. A lane reads back only what it wrote itself, so no barrier is needed.
    __shared__ uint32_t s_nb[kNbBuf][64];
    Kernel kern;
    kern.set(h, dim);
    DensSums S;
    int nb_n = 0;
    auto flush = [&]() {
        const int most = __builtin_amdgcn_readfirstlane((int)wave_max_i(nb_n));
        Neighbour next{};
        if (nb_n > 0) next = neighbour_at(a, s_nb[0][lane]);
        for (int e = 0; e < most; ++e) {
            const Neighbour nb = next;
            if (e + 1 < nb_n) next = neighbour_at(a, s_nb[e + 1][lane]);
            if (e < nb_n) {
                double v[kTerms];
                bool inside = false;
                if (density_terms(nb, qx, qy, qz, kern, v, &inside)) {
#pragma unroll
                    for (int c = 0; c < kTerms; ++c) S.s[c] += v[c];
                    if (inside) ++S.n_inside;
                }
            }
        }
        nb_n = 0;
    };

    // (the far targets are listed at the end: no store precedes the walk's reads)
    const uint64_t lanes = __ballot(mine);
    if (lanes == 0) {
        if (far) a.far_list[atomicAdd(a.n_far, 1u)] = (uint32_t)k;
        return;
    }
    const double r2 = h * h; // the search's radius_sq (hydro.cc:50)
#pragma unroll
    for (int c = 0; c < kTerms; ++c) S.s[c] = 0.0;
    S.n_inside = 0;
    // the staged particles against every target: a neighbour's slot is written behind the ones a
    // lane holds, and stays there if it counts (four at a time between checks for room)
    __shared__ SphereLds lds;
    const double r2t = mine ? r2 : -1.0;
    walk_spheres(a.nodes, mine, qx, qy, qz, h, lds, nullptr, [&](int np, auto allowed) {
        for (int e0 = 0; e0 < np; e0 += 4) {
            if (__ballot(nb_n > kNbBuf - 4) != 0) flush();
            auto test4 = [&](auto ok) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int e = e0 + j; // (up to 63: entries past np are not counted)
                    const double4 q = lds.p[e];
                    const double ex = q.x - qx, ey = q.y - qy, ez = q.z - qz;
                    const bool in = ex * ex + ey * ey + ez * ez < r2t && e < np && ok(e);
                    s_nb[nb_n][lane] = lds.id[e];
                    nb_n += in ? 1 : 0;
                }
            };
            if (allowed.all) test4([](int) { return true; });
            else test4(allowed);
        }
    });
    flush();
    if (mine) density_update(a, k, t, p, h, it, S);
    if (far) a.far_list[atomicAdd(a.n_far, 1u)] = (uint32_t)k;
}

// Whether each slot's particle is gas.
__global__ __launch_bounds__(256) void k_density_gas(size_t nl, const uint32_t* __restrict__ order,
                                                     const uint8_t* __restrict__ type,
                                                     uint8_t* __restrict__ gas) {
    const size_t r = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (r < nl) gas[r] = type[order[r]] == 0 ? 1 : 0;
}

// Start state: every target active at its first guess; a target outside the particle set flags
// status bit 0 (the call then fails before any search).
__global__ __launch_bounds__(256) void k_density_init(int nt, const uint32_t* __restrict__ targets,
                                                      size_t n, const double* __restrict__ h_start,
                                                      double h_default, double* __restrict__ h,
                                                      double* __restrict__ h_lo,
                                                      double* __restrict__ h_hi,
                                                      int* __restrict__ iter,
                                                      uint32_t* __restrict__ act,
                                                      int* __restrict__ status) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    if (targets[t] >= n) atomicOr(status, 1);
    h[t] = h_start ? h_start[t] : h_default;
    h_lo[t] = 0.0;
    h_hi[t] = 0.0;
    iter[t] = 0;
    act[t] = (uint32_t)t;
}

// The far targets' entries in the active list: their target positions.
__global__ __launch_bounds__(256) void k_density_far_act(int nf, const uint32_t* __restrict__ far,
                                                         const uint32_t* __restrict__ act,
                                                         uint32_t* __restrict__ far_act) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < nf) far_act[j] = act[far[j]];
}

// The far targets' keep flags back into the active list's.
__global__ __launch_bounds__(256) void k_density_far_keep(int nf, const uint32_t* __restrict__ far,
                                                          const uint32_t* __restrict__ far_keep,
                                                          uint32_t* __restrict__ keep) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < nf) keep[far[j]] = far_keep[j];
}

// next[j] = cur[pos[j]] for the kept entries (pos from the flags' scan).
__global__ __launch_bounds__(256) void k_density_compact(int nk, const int* __restrict__ pos,
                                                         const uint32_t* __restrict__ cur,
                                                         uint32_t* __restrict__ next) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < nk) next[j] = cur[pos[j]];
}

// The bounding box of all particles (hydro.cc:172-178), as order-preserving 64-bit keys of the
// doubles: min x y z in box[0..2], max in box[3..5] (the max stored complemented so that both
// are atomicMin).
__device__ __forceinline__ unsigned long long dkey(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__global__ __launch_bounds__(256) void k_density_bbox(size_t n, const double* __restrict__ x,
                                                      const double* __restrict__ y,
                                                      const double* __restrict__ z,
                                                      unsigned long long* __restrict__ box) {
    unsigned long long lo[3] = {~0ull, ~0ull, ~0ull}, hi[3] = {~0ull, ~0ull, ~0ull};
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const double v[3] = {x[i], y[i], z[i]};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const unsigned long long kk = dkey(v[d]);
            lo[d] = min(lo[d], kk);
            hi[d] = min(hi[d], ~kk);
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        for (int s = 32; s >= 1; s >>= 1) {
            lo[d] = min(lo[d], (unsigned long long)__shfl_xor((long long)lo[d], s));
            hi[d] = min(hi[d], (unsigned long long)__shfl_xor((long long)hi[d], s));
        }
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            atomicMin(&box[d], lo[d]);
            atomicMin(&box[3 + d], hi[d]);
        }
    }
}

double key_to_double(unsigned long long k) {
    const unsigned long long b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
    double v;
    std::memcpy(&v, &b, sizeof v);
    return v;
}

} // namespace
} // namespace gz

using namespace gz;

extern "C" gz_status gz_tree_density(gz_ctx* ctx, const gz_tree* tree, const gz_particles* p,
                                     const uint32_t* targets, size_t n_t, double des_ngb,
                                     double ngb_tol, const double* h_start, int n_dims,
                                     const double* cond_prev, double tau, double* h, double* rho,
                                     int* nngb, int* iters) {
    clear_error();
    if (!ctx || !tree || !p) return fail(GZ_ERR_INVALID, "gz_tree_density: null argument");
    GZ_HIP(hipSetDevice(ctx->device));
    if (n_t == 0) return GZ_OK;
    if (!targets || !h || !rho || !nngb || !iters || !p->x || !p->y || !p->z || !p->m)
        return fail(GZ_ERR_INVALID, "gz_tree_density: null array");
    if (n_dims < 1 || n_dims > 3)
        return fail(GZ_ERR_INVALID, "gz_tree_density: n_dims=%d (1, 2 or 3)", n_dims);
    if (!(des_ngb > 0) || !(ngb_tol >= 0))
        return fail(GZ_ERR_INVALID, "gz_tree_density: des_ngb must be > 0 and ngb_tol >= 0");
    if (n_t >= 0x7FFFFFFFull) return fail(GZ_ERR_INVALID, "gz_tree_density: n_t too large");
    if (p->n != tree->n)
        return fail(GZ_ERR_INVALID, "gz_tree_density: %zu particles, the tree holds %zu", p->n,
                    (size_t)tree->n);
    hipStream_t st = ctx->stream;
    const int nt = (int)n_t;

    // state: h_lo, h_hi (doubles); iter, the active list, the compaction's output, the keep
    // flags, their scan and the kept positions; the targets' slots and the sort's keys and
    // values (twice); the box keys, the scan total and the status words; the scan's temporary
    // space
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t o = off;
        off += (bytes + 255) & ~size_t(255);
        return o;
    };
    // Many targets: the particles' live values are put in slot order first, where the targets of a
    // wave find their neighbours together (a neighbour's four values cost four scattered reads
    // otherwise, several times a call)
    bool by_slot = n_t >= tree->n_live / 8;
    const size_t o_lo = take(n_t * 8), o_hi = take(n_t * 8), o_iter = take(n_t * 4),
                 o_act = take(n_t * 4), o_nxt = take(n_t * 4), o_keep = take((n_t + 1) * 4),
                 o_scan = take((n_t + 1) * 4), o_kept = take((n_t + 1) * 4),
                 o_slot = take(n_t * 4), o_k0 = take(n_t * 8), o_k1 = take(n_t * 8),
                 o_v0 = take(n_t * 4), o_v1 = take(n_t * 4), o_far = take(n_t * 4),
                 o_fact = take(n_t * 4), o_fkeep = take(n_t * 4),
                 o_srec = take((size_t)std::max(tree->nnodes, 1) * sizeof(SRec)),
                 o_misc = take(256), o_tmp = take(scan_tmp_bytes(n_t + 1)), need = off,
                 o_live = take(by_slot ? tree->n_live * sizeof(double4) : 0),
                 o_gas = take(by_slot && p->type ? tree->n_live : 0);
    DevMem& mem = ctx->scratch[13];
    ScratchUse mem_use(mem);
    by_slot = by_slot && mem.offer(off); // (without the memory for it: through orderbuf)
    GZ_TRY(mem.reserve(need));
    uint8_t* base = mem.as<uint8_t>();
    double* d_lo = reinterpret_cast<double*>(base + o_lo);
    double* d_hi = reinterpret_cast<double*>(base + o_hi);
    int* d_iter = reinterpret_cast<int*>(base + o_iter);
    uint32_t* d_act = reinterpret_cast<uint32_t*>(base + o_act);
    uint32_t* d_nxt = reinterpret_cast<uint32_t*>(base + o_nxt);
    uint32_t* d_keep = reinterpret_cast<uint32_t*>(base + o_keep);
    uint32_t* d_scan = reinterpret_cast<uint32_t*>(base + o_scan);
    int* d_kept = reinterpret_cast<int*>(base + o_kept);
    unsigned long long* d_box = reinterpret_cast<unsigned long long*>(base + o_misc);
    uint32_t* d_total = reinterpret_cast<uint32_t*>(base + o_misc + 64);
    int* d_status = reinterpret_cast<int*>(base + o_misc + 128);
    int* d_sort = reinterpret_cast<int*>(base + o_misc + 192); // bit 1: bad index; [1]: unsorted
    uint32_t* d_nfar = reinterpret_cast<uint32_t*>(base + o_misc + 224);
    int* d_moved = reinterpret_cast<int*>(base + o_misc + 240);
    uint32_t* d_far = reinterpret_cast<uint32_t*>(base + o_far);
    uint32_t* d_fact = reinterpret_cast<uint32_t*>(base + o_fact);
    uint32_t* d_fkeep = reinterpret_cast<uint32_t*>(base + o_fkeep);
    GZ_TRY(fill_zero_u32(reinterpret_cast<uint32_t*>(base + o_misc), 64, st));

    // the default first guess: des_ngb particles at the mean density of the bounding box of all
    // particles (hydro.cc:168-186), the box reduced on the device and the guess formed here
    double h_default = 0.0;
    if (!h_start) {
        if (p->n == 0) return fail(GZ_ERR_INVALID, "gz_tree_density: no particles");
        const unsigned long long init[6] = {~0ull, ~0ull, ~0ull, ~0ull, ~0ull, ~0ull};
        GZ_HIP(hipMemcpyAsync(d_box, init, sizeof init, hipMemcpyHostToDevice, st));
        const unsigned gb = (unsigned)std::min<size_t>(1024, (p->n + 255) / 256);
        k_density_bbox<<<gb, 256, 0, st>>>(p->n, p->x, p->y, p->z, d_box);
        GZ_HIP(hipGetLastError());
        unsigned long long kb[6];
        GZ_HIP(hipMemcpyAsync(kb, d_box, sizeof kb, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        double lo[3], hi[3];
        for (int d = 0; d < 3; ++d) {
            lo[d] = key_to_double(kb[d]);
            hi[d] = key_to_double(~kb[3 + d]);
        }
        const double bbox_volume = (hi[0] - lo[0]) * (hi[1] - lo[1]) * (hi[2] - lo[2]);
        const double np = (double)p->n;
        h_default = std::cbrt(3.0 * des_ngb * bbox_volume / (4.0 * kPi * np));
        if (n_dims == 1) h_default = 0.5 * des_ngb * (hi[0] - lo[0]) / np;
        if (n_dims == 2)
            h_default = std::sqrt(des_ngb * (hi[0] - lo[0]) * (hi[1] - lo[1]) / (kPi * np));
    }
    k_density_init<<<(unsigned)((n_t + 255) / 256), 256, 0, st>>>(
        nt, targets, p->n, h_start, h_default, h, d_lo, d_hi, d_iter, d_act, d_status);
    GZ_HIP(hipGetLastError());
    // the targets' sorted slots: a list out of slot order is walked in slot order (the waves'
    // targets are then neighbours), the results staying by list position
    uint64_t* k0 = reinterpret_cast<uint64_t*>(base + o_k0);
    uint64_t* k1 = reinterpret_cast<uint64_t*>(base + o_k1);
    uint32_t* v0 = reinterpret_cast<uint32_t*>(base + o_v0);
    uint32_t* v1 = reinterpret_cast<uint32_t*>(base + o_v1);
    GZ_TRY(launch_pt_keys(targets, n_t, tree, p->n, reinterpret_cast<int*>(base + o_slot), k0, v0,
                          d_sort, st));
    int head[3] = {0, 0, 0};
    GZ_HIP(hipMemcpyAsync(head, d_status, sizeof(int), hipMemcpyDeviceToHost, st));
    GZ_HIP(hipMemcpyAsync(head + 1, d_sort, 2 * sizeof(int), hipMemcpyDeviceToHost, st));
    GZ_HIP(hipStreamSynchronize(st));
    if ((head[0] & 1) || (head[1] & 2))
        return fail(GZ_ERR_INVALID, "gz_tree_density: a target is outside the particle set");
    if (head[2]) {
        int bits = 1;
        while (bits < 40 && (1ull << bits) <= (unsigned long long)tree->n_live) ++bits;
        GZ_TRY(radix_sort_pairs(k0, v0, k1, v1, n_t, bits, ctx->scratch[3], st));
        GZ_HIP(hipMemcpyAsync(d_act, v0, n_t * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
    }
    if (tree->depth + 2 > kPtDepth)
        return fail(GZ_ERR_INTERNAL, "gz_tree_density: tree depth %d exceeds the walk's stack",
                    tree->depth);

    DensArgs a{};
    a.targets = targets;
    a.x = p->x;
    a.y = p->y;
    a.z = p->z;
    a.m = p->m;
    a.type = p->type;
    a.des_ngb = des_ngb;
    a.ngb_tol = ngb_tol;
    a.n_dims = n_dims;
    a.cond_prev = cond_prev;
    a.h = h;
    a.h_lo = d_lo;
    a.h_hi = d_hi;
    a.rho = rho;
    a.iter = d_iter;
    a.nngb = nngb;
    a.iters = iters;
    a.keep = d_keep;
    a.tslot = reinterpret_cast<const int*>(base + o_slot);
    a.slot_leaf = tree->slot_leaf;
    a.far_list = d_far;
    a.n_far = d_nfar;
    GZ_TRY(launch_sphere_nodes(tree, tau, reinterpret_cast<SRec*>(base + o_srec), d_moved,
                               &a.nodes, st));
    if (by_slot && tree->n_live > 0) {
        GZ_TRY(gather_live(ctx, p, tree, reinterpret_cast<double4*>(base + o_live)));
        a.live = reinterpret_cast<const double4*>(base + o_live);
        if (p->type) {
            k_density_gas<<<(unsigned)((tree->n_live + 255) / 256), 256, 0, st>>>(
                tree->n_live, tree->orderbuf, p->type, base + o_gas);
            GZ_HIP(hipGetLastError());
            a.live_gas = base + o_gas;
        }
    }
    a.wn = tree->wn;
    a.size = tree->size;
    a.src = tree->src;
    a.orderbuf = tree->orderbuf;

    const double cand = des_ngb * near_volume(1.0, n_dims); // a converged target's candidates
    const bool collect = cand <= kCollectMax;
    const uint32_t last = (cand <= kCollectMost) ? kLastTargets : kLastTargetsFull;
    // rounds: a target takes at most 100 steps and one last search
    uint32_t n_act = (uint32_t)n_t;
    for (int round = 0; n_act > 0; ++round) {
        if (round > kMaxIter + 1)
            return fail(GZ_ERR_INTERNAL, "gz_tree_density: the solve did not end");
        a.act = d_act;
        a.n_act = (int)n_act;
        const bool loop = n_act <= last; // to the end in one launch
        GZ_TRY(fill_zero_u32(d_nfar, 1, st));
        if (!loop) k_density_round<<<(n_act + 63) / 64, 64, 0, st>>>(a);
        else if (!collect) k_density_far<true><<<n_act, 64, 0, st>>>(a);
        else if (n_act <= kNearFar) k_density_near<true><<<n_act, 64, 0, st>>>(a);
        else k_density_near<false><<<n_act, 64, 0, st>>>(a);
        GZ_HIP(hipGetLastError());
        if (loop && (!collect || n_act <= kNearFar)) break;
        uint32_t n_far = 0;
        GZ_HIP(hipMemcpyAsync(&n_far, d_nfar, sizeof n_far, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        if (n_far > 0) {
            // the far targets: a wave each, in the round's order (their keep flags are then
            // moved to the round's positions)
            const unsigned gf = (n_far + 255) / 256;
            k_density_far_act<<<gf, 256, 0, st>>>((int)n_far, d_far, d_act, d_fact);
            GZ_HIP(hipGetLastError());
            DensArgs f = a;
            f.act = d_fact;
            f.n_act = (int)n_far;
            f.keep = d_fkeep;
            if (loop) k_density_far<true><<<n_far, 64, 0, st>>>(f);
            else k_density_far<false><<<n_far, 64, 0, st>>>(f);
            GZ_HIP(hipGetLastError());
            if (loop) break; // every target is done
            k_density_far_keep<<<gf, 256, 0, st>>>((int)n_far, d_far, d_fkeep, d_keep);
            GZ_HIP(hipGetLastError());
        }
        if (loop) break;
        // the targets still active, in their order: kept positions, then their target indices
        GZ_TRY(exclusive_scan_u32(d_keep, d_scan, n_act, d_total, base + o_tmp, st, d_kept));
        uint32_t n_next = 0;
        GZ_HIP(hipMemcpyAsync(&n_next, d_total, sizeof n_next, hipMemcpyDeviceToHost, st));
        GZ_HIP(hipStreamSynchronize(st));
        if (n_next > 0) {
            k_density_compact<<<(n_next + 255) / 256, 256, 0, st>>>((int)n_next, d_kept, d_act,
                                                                     d_nxt);
            GZ_HIP(hipGetLastError());
            std::swap(d_act, d_nxt);
        }
        n_act = n_next;
    }
    GZ_HIP(hipStreamSynchronize(st));
    return GZ_OK;
}
