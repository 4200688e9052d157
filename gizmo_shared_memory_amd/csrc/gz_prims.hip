// Device-wide primitives: an exclusive scan and a stable LSD radix sort of (64-bit key, 32-bit value)
// pairs. Both are memory-bound at the sizes of large trees (>= 1M
// keys), where one launch has a thousand workgroups, and bound by their launches below that.
#include <algorithm>

#include "gz_internal.h"
#include "gz_wave.h"

namespace gz {

// ---- wave / block scans ----------------------------------------------------------------------
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t x) {
    return wave_incl_scan_dpp(x);
}

// Exclusive scan across a 256-thread block (4 waves). s4 is a 4-entry LDS scratch.
__device__ __forceinline__ uint32_t block256_exclusive_scan(uint32_t v, uint32_t* s4,
                                                            uint32_t& total) {
    const uint32_t inc = wave_inclusive_scan(v);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 63) s4[w] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t s = s4[k];
        off += (k < w) ? s : 0u;
        tot += s;
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

constexpr int kScanThreads = 256;
constexpr int kScanIpt = 8;
constexpr int kScanTile = kScanThreads * kScanIpt;

__global__ __launch_bounds__(kScanThreads) void k_scan_partials(const uint32_t* __restrict__ in,
                                                                size_t n,
                                                                uint32_t* __restrict__ partial) {
    __shared__ uint32_t s4[4];
    const size_t base = (size_t)blockIdx.x * kScanTile;
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kScanIpt; ++j) {
        const size_t i = base + (size_t)j * kScanThreads + threadIdx.x;
        if (i < n) sum += in[i];
    }
    uint32_t total;
    (void)block256_exclusive_scan(sum, s4, total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// One workgroup of 1024 threads scans the per-tile partial sums in place, chunk by chunk.
__global__ __launch_bounds__(1024) void k_scan_partials_scan(uint32_t* __restrict__ partial,
                                                             size_t nb,
                                                             uint32_t* __restrict__ total_out) {
    __shared__ uint32_t s16[16];
    __shared__ uint32_t s_carry;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (size_t base = 0; base < nb; base += 1024) {
        const size_t i = base + threadIdx.x;
        const uint32_t v = (i < nb) ? partial[i] : 0u;
        const uint32_t inc = wave_inclusive_scan(v);
        if (lane == 63) s16[w] = inc;
        __syncthreads();
        uint32_t off = 0, tot = 0;
        for (int k = 0; k < 16; ++k) {
            const uint32_t s = s16[k];
            off += (k < w) ? s : 0u;
            tot += s;
        }
        const uint32_t carry = s_carry;
        if (i < nb) partial[i] = carry + off + inc - v;
        __syncthreads();
        if (threadIdx.x == 0) s_carry = carry + tot;
        __syncthreads();
    }
    if (threadIdx.x == 0 && total_out) *total_out = s_carry;
}

// starts (optional): for a scan of 0/1 flags, starts[out[i]] = i wherever in[i] is set (the
// first index of each run that the flags open).
__global__ __launch_bounds__(kScanThreads) void k_scan_apply(const uint32_t* in, uint32_t* out,
                                                             size_t n,
                                                             const uint32_t* __restrict__ partial,
                                                             int* __restrict__ starts, int vec) {
    __shared__ uint32_t s4[4];
    // blocked arrangement: thread t owns elements base + t*kScanIpt .. + kScanIpt - 1, read and
    // written as two 16-byte vectors when the tile is whole and the arrays are aligned
    const size_t base = (size_t)blockIdx.x * kScanTile + (size_t)threadIdx.x * kScanIpt;
    const bool whole = vec && base + kScanIpt <= n;
    uint32_t v[kScanIpt];
    if (whole) {
        const uint4 a = reinterpret_cast<const uint4*>(in + base)[0];
        const uint4 b = reinterpret_cast<const uint4*>(in + base)[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int j = 0; j < kScanIpt; ++j) v[j] = (base + j < n) ? in[base + j] : 0u;
    }
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kScanIpt; ++j) sum += v[j];
    uint32_t total;
    uint32_t run = block256_exclusive_scan(sum, s4, total) + partial[blockIdx.x];
    uint32_t o[kScanIpt];
#pragma unroll
    for (int j = 0; j < kScanIpt; ++j) {
        o[j] = run;
        if (starts && v[j] && base + j < n) starts[run] = (int)(base + j);
        run += v[j];
    }
    if (whole) {
        reinterpret_cast<uint4*>(out + base)[0] = make_uint4(o[0], o[1], o[2], o[3]);
        reinterpret_cast<uint4*>(out + base)[1] = make_uint4(o[4], o[5], o[6], o[7]);
    } else {
#pragma unroll
        for (int j = 0; j < kScanIpt; ++j)
            if (base + j < n) out[base + j] = o[j];
    }
}

// One workgroup scans the whole array: below kScanSmall elements two more launches cost more than
// the chip's width gains (a level of the tree build, a pass of a small sort).
constexpr size_t kScanSmall = 16384;
__global__ __launch_bounds__(1024) void k_scan_small(const uint32_t* in, uint32_t* out, int n,
                                                     uint32_t* __restrict__ total_out,
                                                     int* __restrict__ starts) {
    __shared__ uint32_t s16[16];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t carry = 0;
    for (int base = 0; base < n; base += 1024 * kScanIpt) {
        const int i0 = base + threadIdx.x * kScanIpt;
        uint32_t v[kScanIpt], sum = 0;
#pragma unroll
        for (int j = 0; j < kScanIpt; ++j) {
            v[j] = (i0 + j < n) ? in[i0 + j] : 0u;
            sum += v[j];
        }
        const uint32_t inc = wave_inclusive_scan(sum);
        if (lane == 63) s16[w] = inc;
        __syncthreads();
        uint32_t off = 0, tot = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const uint32_t s = s16[k];
            off += (k < w) ? s : 0u;
            tot += s;
        }
        uint32_t run = carry + off + inc - sum;
#pragma unroll
        for (int j = 0; j < kScanIpt; ++j) {
            if (i0 + j < n) {
                out[i0 + j] = run;
                if (starts && v[j]) starts[run] = i0 + j;
            }
            run += v[j];
        }
        carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0 && total_out) *total_out = carry;
}

size_t scan_tmp_bytes(size_t n) {
    const size_t nb = (n + kScanTile - 1) / kScanTile;
    return (nb + 64) * sizeof(uint32_t);
}

gz_status exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t n, uint32_t* total_dev,
                             void* tmp, hipStream_t st, int* starts) {
    if (n == 0) {
        if (total_dev) GZ_HIP(hipMemsetAsync(total_dev, 0, sizeof(uint32_t), st));
        return GZ_OK;
    }
    if (n <= kScanSmall) {
        k_scan_small<<<1, 1024, 0, st>>>(in, out, (int)n, total_dev, starts);
        GZ_HIP(hipGetLastError());
        return GZ_OK;
    }
    const size_t nb = (n + kScanTile - 1) / kScanTile;
    uint32_t* partial = static_cast<uint32_t*>(tmp);
    k_scan_partials<<<(unsigned)nb, kScanThreads, 0, st>>>(in, n, partial);
    k_scan_partials_scan<<<1, 1024, 0, st>>>(partial, nb, total_dev);
    const int vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    k_scan_apply<<<(unsigned)nb, kScanThreads, 0, st>>>(in, out, n, partial, starts, vec);
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}

__global__ __launch_bounds__(256) void k_fill_zero_u32(uint32_t* __restrict__ a, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) a[i] = 0u;
}

gz_status fill_zero_u32(uint32_t* a, size_t n, hipStream_t st) {
    if (n == 0) return GZ_OK;
    k_fill_zero_u32<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(a, n);
    GZ_HIP(hipGetLastError());
    return GZ_OK;
}

// ---- radix sort ------------------------------------------------------------------------------
// Stable LSD passes of 8 bits, each a count of every tile's digits and a scatter. A tile's wave
// ranks its own contiguous elements against counters of its own (no barrier between them), the
// tile is put in digit order in LDS, and the runs of equal digits are then written out by
// neighbouring lanes.
constexpr int kRsThreads = 256;
constexpr int kRsRadix = 256;
// Tiles: 4096 elements make runs of 16 (128 B of keys) on average; below kRsBig elements smaller
// tiles keep more of the chip busy, and up to kRsDirect tiles each scatter workgroup adds up the
// counts of the tiles before it instead of waiting for a scan.
constexpr size_t kRsBig = size_t(1) << 20;
constexpr uint32_t kRsDirect = 128;

// Digit counts of every tile: hist[d * nb + b], or hist[b * 256 + d] for the direct scatter.
template <int IPT>
__global__ __launch_bounds__(kRsThreads) void k_rs_count(const uint64_t* __restrict__ keys,
                                                         size_t n, int shift, uint32_t nb,
                                                         int direct,
                                                         uint32_t* __restrict__ hist) {
    __shared__ uint32_t c[kRsRadix];
    c[threadIdx.x] = 0;
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * (kRsThreads * IPT);
    uint32_t d[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        const size_t i = base + (size_t)j * kRsThreads + threadIdx.x;
        d[j] = (i < n) ? (uint32_t)(keys[i] >> shift) & 255u : 256u;
    }
#pragma unroll
    for (int j = 0; j < IPT; ++j)
        if (d[j] < 256u) atomicAdd(&c[d[j]], 1u);
    __syncthreads();
    const size_t at = direct ? (size_t)blockIdx.x * kRsRadix + threadIdx.x
                             : (size_t)threadIdx.x * nb + blockIdx.x;
    hist[at] = c[threadIdx.x];
}

template <int IPT>
__global__ __launch_bounds__(kRsThreads) void k_rs_scatter(
    const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint64_t* __restrict__ kout, uint32_t* __restrict__ vout, size_t n, int shift, uint32_t nb,
    int direct, const uint32_t* __restrict__ offs) {
    constexpr int kTile = kRsThreads * IPT;
    __shared__ uint64_t s_key[kTile];
    __shared__ uint32_t s_val[kTile];
    __shared__ uint32_t s_cnt[4][kRsRadix]; // a wave's count so far, then its first place
    __shared__ uint32_t s_goff[kRsRadix];   // output place of a digit's run, less its place here
    __shared__ uint32_t s4[4];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const size_t base = (size_t)blockIdx.x * kTile;
    const int count = (int)((n - base < (size_t)kTile) ? n - base : (size_t)kTile);
    // element (w, j, lane) of the tile: the input order is w, then j, then lane
    uint64_t key[IPT];
    uint32_t val[IPT], rank[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        const int e = (w * IPT + j) * kWave + lane;
        key[j] = 0;
        val[j] = 0;
        if (e < count) {
            key[j] = kin[base + e];
            val[j] = vin[base + e];
        }
    }
    // where this tile's digits go: thread d's digit, after the lower digits of all tiles and its
    // own digit of the tiles before
    uint32_t gplace, total;
    if (direct) {
        uint32_t before = 0, all = 0;
#pragma unroll 8
        for (uint32_t b = 0; b < nb; ++b) {
            const uint32_t c = offs[(size_t)b * kRsRadix + tid];
            before += (b < blockIdx.x) ? c : 0u;
            all += c;
        }
        gplace = block256_exclusive_scan(all, s4, total) + before;
    } else {
        gplace = offs[(size_t)tid * nb + blockIdx.x];
    }
    for (int k = lane; k < kRsRadix; k += kWave) s_cnt[w][k] = 0;
    __syncthreads();
    const uint64_t below_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        const bool valid = (w * IPT + j) * kWave + lane < count;
        const uint32_t d = (uint32_t)(key[j] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool set = (d >> bit) & 1u;
            const uint64_t m = __ballot(set);
            peers &= set ? m : ~m;
        }
        const uint32_t below = (uint32_t)__popcll(peers & below_mask);
        // the wave's own counter: read by every peer, then advanced by the first of them (LDS
        // accesses of one wave stay in order)
        volatile uint32_t* c = &s_cnt[w][d];
        const uint32_t old = *c;
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) *c = old + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rank[j] = old + below;
    }
    __syncthreads();
    uint32_t c[4], mine = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        c[k] = s_cnt[k][tid];
        mine += c[k];
    }
    uint32_t place = block256_exclusive_scan(mine, s4, total);
    s_goff[tid] = gplace - place;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        s_cnt[k][tid] = place;
        place += c[k];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        if ((w * IPT + j) * kWave + lane < count) {
            const uint32_t d = (uint32_t)(key[j] >> shift) & 255u;
            const uint32_t at = s_cnt[w][d] + rank[j];
            s_key[at] = key[j];
            s_val[at] = val[j];
        }
    }
    __syncthreads();
    for (int e = tid; e < count; e += kRsThreads) {
        const uint64_t k = s_key[e];
        const uint32_t pos = s_goff[(uint32_t)(k >> shift) & 255u] + (uint32_t)e;
        kout[pos] = k;
        vout[pos] = s_val[e];
    }
}

gz_status radix_sort_pairs(uint64_t*& keys, uint32_t*& vals, uint64_t*& keys_alt,
                           uint32_t*& vals_alt, size_t n, int bits, DevMem& scratch,
                           hipStream_t st) {
    if (n <= 1) return GZ_OK;
    if (n >= 0xFFFFFFFFull) return fail(GZ_ERR_INVALID, "radix sort: %zu keys exceed 2^32-1", n);
    const int npasses = std::min(8, (bits + 7) / 8);
    const bool big = n >= kRsBig;
    const size_t tile = (size_t)kRsThreads * (big ? 16 : 8);
    const uint32_t nb = (uint32_t)((n + tile - 1) / tile);
    const int direct = nb <= kRsDirect;
    const size_t hist_n = (size_t)kRsRadix * nb;
    const size_t hist_bytes = (hist_n * sizeof(uint32_t) + 255) & ~size_t(255);
    GZ_TRY(scratch.reserve(hist_bytes + scan_tmp_bytes(hist_n) + 256));
    uint32_t* hist = scratch.as<uint32_t>();
    void* scan_tmp = scratch.as<uint8_t>() + hist_bytes;
    for (int p = 0; p < npasses; ++p) {
        const int shift = 8 * p;
        if (big) k_rs_count<16><<<nb, kRsThreads, 0, st>>>(keys, n, shift, nb, direct, hist);
        else k_rs_count<8><<<nb, kRsThreads, 0, st>>>(keys, n, shift, nb, direct, hist);
        GZ_HIP(hipGetLastError());
        if (!direct) GZ_TRY(exclusive_scan_u32(hist, hist, hist_n, nullptr, scan_tmp, st));
        if (big)
            k_rs_scatter<16><<<nb, kRsThreads, 0, st>>>(keys, vals, keys_alt, vals_alt, n, shift,
                                                        nb, direct, hist);
        else
            k_rs_scatter<8><<<nb, kRsThreads, 0, st>>>(keys, vals, keys_alt, vals_alt, n, shift,
                                                       nb, direct, hist);
        GZ_HIP(hipGetLastError());
        std::swap(keys, keys_alt);
        std::swap(vals, vals_alt);
    }
    return GZ_OK;
}

} // namespace gz
