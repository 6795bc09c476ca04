// bands.h -- index arithmetic of dense grids and the compaction of narrow bands, shared by
// the liquid-step kernels (liquid.hip, redist.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace shk {

// (i, j, k) of a linear index with 32-bit unsigned arithmetic (shk_create bounds the
// cells by 2^31, so every face array has fewer than 2^32 entries)
// Exact division of a 32-bit index by an extent n without a divide sequence:
// floor(q / n) = floor(m q / 2^64) with m = ceil(2^64 / n) for every 32-bit q and
// 2 <= n < 2^32 (Lemire, Kaser and Kurz, "Faster remainder by direct computation",
// 2019).  m is computed on the host; n = 1 takes q itself.
struct Div32 {
    uint32_t n;
    uint64_t m;
};
inline Div32 div32(int n) { return Div32{(uint32_t)n, n > 1 ? ~0ull / (uint64_t)n + 1 : 0ull}; }
__device__ inline uint32_t quot(uint32_t q, Div32 d) {
    return d.n > 1 ? (uint32_t)__umul64hi(d.m, (uint64_t)q) : q;
}

// the x and y extents of an index space (a face or cell array), for decompose
struct Split {
    Div32 x, y;
};

__device__ inline void decompose(int64_t q, Split sp, int &i, int &j, int &k) {
    const uint32_t u = (uint32_t)q;
    const uint32_t t = quot(u, sp.x);
    i = (int)(u - t * sp.x.n);
    k = (int)quot(t, sp.y);
    j = (int)(t - (uint32_t)k * sp.y.n);
}

constexpr int kBandNT = 256;

// Sum of a per-thread count over a block of kBandNT threads, valid in thread 0.
__device__ inline unsigned int block_count(unsigned int v) {
    __shared__ unsigned int w[kBandNT / 64];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned int t = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < kBandNT / 64; ++i) t += w[i];
    return t;
}

// A band holds a few percent of the cells: the passes over it run on a list of its cells
// instead of one thread per cell of the grid (256^3: 65,536 workgroups that mostly read one
// byte and leave, 55..100 us per pass).  Each block compacts 4096 cells, in order, into a
// range that one atomic reserves; the ranges' order does not matter, every cell of a pass
// being independent.  *count starts at 0.  vec: mask is 16-byte aligned.  The list has room
// for every cell (4 bytes each, 0.5 GB at 512^3), a band of any width being allowed.
//
// A wide band is better left where it lies: writing its list takes 113 us for the 16.8 million
// cells of 256^3, the ranges come in the order in which blocks arrive, and a pass over them
// shares fewer planes in the caches (level-set advection, list / all cells by their mask: all in
// the band 1187 / 623 us, a quarter 337 / 229, a tenth 159 / 150).  With wide > 0 every block
// looks at the same kBandNT cells, and where more than `wide` of them are in the band it says so
// by a count of kBandWide and leaves the list alone.
constexpr unsigned int kBandWide = 0xffffffffu;
constexpr int kBandWideOf256 = 43;  // a sixth
__global__ __launch_bounds__(kBandNT) inline void k_band_list(int64_t n, const uint8_t *__restrict__ mask, int vec,
                                                              int wide, uint32_t *__restrict__ list,
                                                              unsigned int *__restrict__ count) {
    if (wide) {
        // multiples of the golden ratio: spread evenly over any stretch of the grid
        const uint64_t at = ((uint64_t)(threadIdx.x * 2654435769u) * (uint64_t)n) >> 32;
        if (__syncthreads_count(mask[at] != 0) > wide) {
            if (blockIdx.x == 0 && threadIdx.x == 0) *count = kBandWide;
            return;
        }
    }
    const int64_t c0 = blockIdx.x * (int64_t)(16 * kBandNT) + 16 * (int64_t)threadIdx.x;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    if (vec && c0 + 16 <= n) {
        const uint4 v = *reinterpret_cast<const uint4 *>(mask + c0);
        w[0] = v.x;
        w[1] = v.y;
        w[2] = v.z;
        w[3] = v.w;
    } else {
        for (int q = 0; q < 16; ++q)
            if (c0 + q < n) w[q >> 2] |= (uint32_t)mask[c0 + q] << (8 * (q & 3));
    }
    unsigned int bits = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) bits |= ((w[q >> 2] >> (8 * (q & 3))) & 0xffu ? 1u : 0u) << q;
    // exclusive prefix of the counts over the block
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned int own = __popc(bits);
    unsigned int inc = own;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int u = __shfl_up(inc, o, 64);
        if (lane >= o) inc += u;
    }
    __shared__ unsigned int wtot[kBandNT / 64], base;
    if (lane == 63) wtot[wave] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned int t = 0;
        for (int i = 0; i < kBandNT / 64; ++i) t += wtot[i];
        base = t ? atomicAdd(count, t) : 0u;
    }
    __syncthreads();
    unsigned int at = base + inc - own;
    for (int i = 0; i < wave; ++i) at += wtot[i];
    while (bits) {
        const int q = __ffs(bits) - 1;
        bits &= bits - 1;
        list[at++] = (uint32_t)(c0 + q);
    }
}
inline unsigned band_list_blocks(int64_t n) { return (unsigned)((n + 16 * kBandNT - 1) / (16 * kBandNT)); }
// blocks of a grid-stride pass over a list whose length only the device knows
constexpr unsigned kBandBlocks = 2048;

// The cells of a pass over a band of n cells with list, *count and mask: all cells by their mask
// where there is no list (count null) or the band is wide.
struct BandPass {
    const uint32_t *list;
    const unsigned int *count;
    const uint8_t *mask;
    uint32_t n;
    // the list's entries, or every cell; wide: whether cell(at) has to be looked up in the mask
    __device__ uint32_t length(bool &wide) const {
        const unsigned int len = count ? *count : kBandWide;
        wide = len == kBandWide;
        return wide ? n : len;
    }
};

__global__ inline void k_zero_counts(unsigned int *p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0u;
}

}  // namespace shk
