// redist.hip -- PDE redistancing of the liquid level set on the GPU: the
// pderedistancer3 plugin's redistance(phi, width) (src/redistancer/pderedistancer3.cpp:
// 39-183) on a dense level set with a per-cell activity mask (the narrow band).
//
// The trim, the dilations and the last step pass over the grid, the initial values and the
// pseudo-time steps over a list of the band's cells, made after the dilations (bands.h): at
// 256^3 the band holds about 4% of the cells, and what bounded the dense passes was not
// memory but their 16.8 million threads, each with a 64-bit index division, most of which
// found nothing to do.  The dense passes take four cells per thread and skip groups without
// work.  The level set evolves in the caller's array and one work array (cells off the band
// keep the caller's values, which carry their side).  256^3 pool+sphere, width 3: the kernels
// of the call 0.95 -> 0.33 ms; its counts went to one address per wave (0.24 ms of it), now
// per block.
//
// Steps:
//   1. trim_narrowband (src/utility/gridutility3.cpp:184-216): an active cell stays active
//      iff an active axis neighbour has the opposite sign, decided on the activity before
//      the trim;
//   2. `width` dilations (pderedistancer3.cpp:50-68, with dilate3.h:43-97's rule that a
//      round reads the state before it): a newly active cell takes -dx or +dx by the sign
//      of its first active neighbour in the order -x, +x, -y, +y, -z, +z;
//   3. the initial level set phi0 and its smoothed sign phi0 / sqrt(phi0^2 + dx^2);
//   4. ceil(width / rate) steps of dphi/dt = sgn0 (1 - |grad phi|) with dt = rate * dx
//      (Euler, or Heun's RK2), the gradient from upwind one-sided differences that use
//      the interface distance (utility::fraction of phi0) across a sign change of phi0
//      (pderedistancer3.cpp:86-134); the updates round as the reference's float arrays do:
//      fl(fl(d * fl(dt)) + phi) (array3.h:889-951);
//   5. cells with |phi| > width*dx leave the band, and every cell off the band takes the
//      level-set fill of its side, -width*dx where its value is negative and +width*dx
//      elsewhere (set_as_levelset + flood_fill, pderedistancer3.cpp:176-182).  The dense
//      layout carries each cell's side in its value, which is what the reference's flood
//      fill reconstructs from the band.
// FP contraction is off: every product and sum rounds as written, as in the reference's
// x86-64 build.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "bands.h"
#include "ctx_internal.h"
#include "shk_fractions.h"

namespace shk {

struct RedistWork {
    DevBuf<uint8_t> m;          // per cell: 0 off the band, else a tag (the round that took it in) and its side
    DevBuf<float> p, phi0, sgn, d0, tmp;
    DevBuf<uint32_t> list;      // the band's cells
    DevBuf<unsigned int> count;  // list length, final band
    void release() {
        m.release();
        list.release();
        p.release();
        phi0.release();
        sgn.release();
        d0.release();
        tmp.release();
        count.release();
    }
};

void redist_destroy(RedistWork *w) {
    if (!w) return;
    w->release();
    delete w;
}

namespace {

struct RShape {
    int nx, ny, nz;
    __host__ __device__ int64_t at(int i, int j, int k) const {
        return (int64_t)i + (int64_t)nx * ((int64_t)j + (int64_t)ny * k);
    }
};

// neighbour t of (i, j, k) in the order -x, +x, -y, +y, -z, +z; false if out of bounds
__device__ inline bool neighbour(const RShape &s, int i, int j, int k, int t, int64_t &e) {
    const int a = t >> 1, d = (t & 1) ? 1 : -1;
    const int ii = i + (a == 0) * d, jj = j + (a == 1) * d, kk = k + (a == 2) * d;
    if (ii < 0 || jj < 0 || kk < 0 || ii >= s.nx || jj >= s.ny || kk >= s.nz) return false;
    e = s.at(ii, jj, kk);
    return true;
}

// A cell of the band carries the tag 1 + the dilation round that took it in (1: the trimmed
// band), with kBelow where its level set is below 0.
constexpr uint8_t kBelow = 0x80;

// four cells per thread: m = 1 (and the side) where the cell stays in the trimmed band
__global__ __launch_bounds__(256) void k_redist_trim(RShape s, Split sp, const float *__restrict__ phi,
                                                     const uint8_t *__restrict__ band, int vec,
                                                     uint8_t *__restrict__ m) {
#pragma clang fp contract(off)
    const int64_t n = (int64_t)s.nx * s.ny * s.nz;
    const int64_t c0 = (blockIdx.x * (int64_t)256 + threadIdx.x) * 4;
    if (c0 >= n) return;
    uint8_t in[4], out[4] = {0, 0, 0, 0};
    if (vec && c0 + 4 <= n) {
        const uchar4 v = *reinterpret_cast<const uchar4 *>(band + c0);
        in[0] = v.x;
        in[1] = v.y;
        in[2] = v.z;
        in[3] = v.w;
    } else {
        for (int q = 0; q < 4; ++q) in[q] = c0 + q < n ? band[c0 + q] : 0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (!in[q]) continue;
        const int64_t c = c0 + q;
        int i, j, k;
        decompose(c, sp, i, j, k);
        const double p = phi[c];
        bool keep = false;
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            int64_t e;
            if (neighbour(s, i, j, k, t, e) && band[e] && p * (double)phi[e] < 0.0) keep = true;
        }
        if (keep) out[q] = 1 | (p < 0.0 ? kBelow : 0);
    }
    // m is padded to a multiple of four
    *reinterpret_cast<uchar4 *>(m + c0) = make_uchar4(out[0], out[1], out[2], out[3]);
}

// One dilation, in place: a cell off the band takes the side of its first neighbour in the
// band before this round.  A cell that this round takes in carries the tag round + 1, which
// its neighbours do not count whether they see it or not.  four cells per thread; rows4: the
// rows are multiples of four, so the group's y and z neighbours are groups of their own
__global__ __launch_bounds__(256) void k_redist_dilate(RShape s, Split sp, int round, int rows4, uint8_t *m) {
    const int64_t n = (int64_t)s.nx * s.ny * s.nz;
    const int64_t c0 = (blockIdx.x * (int64_t)256 + threadIdx.x) * 4;
    if (c0 >= n) return;
    const uchar4 v = *reinterpret_cast<const uchar4 *>(m + c0);
    const uint8_t own[4] = {v.x, v.y, v.z, v.w};
    if (own[0] && own[1] && own[2] && own[3]) return;
    auto counts = [round](uint8_t t) { return t != 0 && (t & ~kBelow) <= round; };
    if (rows4) {
        int i, j, k;
        decompose(c0, sp, i, j, k);
        const int64_t sy = s.nx, sz = (int64_t)s.nx * s.ny;
        const uint8_t xm = i > 0 ? m[c0 - 1] : 0, xp = i + 4 < s.nx ? m[c0 + 4] : 0;
        const uchar4 z4 = make_uchar4(0, 0, 0, 0);
        const uchar4 ym = j > 0 ? *reinterpret_cast<const uchar4 *>(m + c0 - sy) : z4;
        const uchar4 yp = j + 1 < s.ny ? *reinterpret_cast<const uchar4 *>(m + c0 + sy) : z4;
        const uchar4 zm = k > 0 ? *reinterpret_cast<const uchar4 *>(m + c0 - sz) : z4;
        const uchar4 zp = k + 1 < s.nz ? *reinterpret_cast<const uchar4 *>(m + c0 + sz) : z4;
        const uint8_t nb[4][6] = {{xm, own[1], ym.x, yp.x, zm.x, zp.x},
                                  {own[0], own[2], ym.y, yp.y, zm.y, zp.y},
                                  {own[1], own[3], ym.z, yp.z, zm.z, zp.z},
                                  {own[2], xp, ym.w, yp.w, zm.w, zp.w}};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (own[q]) continue;
            uint8_t first = 0;
#pragma unroll
            for (int t = 5; t >= 0; --t)
                if (counts(nb[q][t])) first = nb[q][t];
            if (first) m[c0 + q] = (uint8_t)(round + 1) | (first & kBelow);
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t c = c0 + q;
        if (own[q] || c >= n) continue;
        int i, j, k;
        decompose(c, sp, i, j, k);
        uint8_t first = 0;
#pragma unroll
        for (int t = 5; t >= 0; --t) {
            int64_t e;
            if (neighbour(s, i, j, k, t, e)) {
                const uint8_t nm = m[e];
                if (counts(nm)) first = nm;
            }
        }
        if (first) m[c] = (uint8_t)(round + 1) | (first & kBelow);
    }
}

// the band's initial values: a cell taken in by a dilation starts at -/+ dx
__global__ __launch_bounds__(256) void k_redist_init(double dx, const uint32_t *__restrict__ list,
                                                     const unsigned int *__restrict__ count,
                                                     const uint8_t *__restrict__ m, float *__restrict__ phi,
                                                     float *__restrict__ phi0, float *__restrict__ sgn) {
#pragma clang fp contract(off)
    const unsigned int len = *count;
    for (unsigned int e = blockIdx.x * 256 + threadIdx.x; e < len; e += gridDim.x * 256) {
        const uint32_t c = list[e];
        const uint8_t t = m[c];
        float f = phi[c];
        if ((t & ~kBelow) != 1) phi[c] = f = t & kBelow ? (float)fmin(0.0, 0.0 - dx) : (float)fmax(0.0, 0.0 + dx);
        const double v = f;
        phi0[c] = f;
        sgn[c] = (float)(v / sqrt(v * v + dx * dx));
    }
}

// sgn0 (1 - |grad phi|) at an active cell (pderedistancer3.cpp:86-134)
__device__ inline float redist_rate(const RShape &s, double dx, const float *__restrict__ phi,
                                    const float *__restrict__ phi0, const float *__restrict__ sgn,
                                    const uint8_t *__restrict__ m, int i, int j, int k, int64_t c) {
#pragma clang fp contract(off)
    const double sgn0 = sgn[c];
    const double p0 = phi0[c];
    const double p = phi[c];
    const int ijk[3] = {i, j, k};
    const int ext[3] = {s.nx, s.ny, s.nz};
    const int64_t stride[3] = {1, (int64_t)s.nx, (int64_t)s.nx * s.ny};
    double g2 = 0.0;
    for (int dim = 0; dim < 3; ++dim) {
        int sel = 0;
        const double tmp = sgn0 * p;
        double pb = 0.0, pf = 0.0, g = 0.0;
        const int64_t cb = c - stride[dim], cf = c + stride[dim];
        if (ijk[dim] > 0 && m[cb]) {
            pb = phi[cb];
            if (sgn0 * pb < tmp) sel = -1;
        }
        if (ijk[dim] < ext[dim] - 1 && m[cf]) {
            pf = phi[cf];
            if (sgn0 * pf < tmp) {
                if (sel == 0)
                    sel = 1;
                else if (sgn0 * pf < sgn0 * pb)
                    sel = 1;
            }
        }
        if (sel == -1) {
            const double frac = fraction(p0, (double)phi0[cb]);
            if (frac == 1.0 || frac == 0.0)
                g = (p - pb) / dx;
            else if (sgn0 < 0.0)
                g = p / (dx * frac);
            else
                g = p / (dx * (1.0 - frac));
        } else if (sel == 1) {
            const double frac = fraction(p0, (double)phi0[cf]);
            if (frac == 1.0 || frac == 0.0)
                g = (pf - p) / dx;
            else if (sgn0 < 0.0)
                g = -p / (dx * frac);
            else
                g = -p / (dx * (1.0 - frac));
        }
        // |grad|^2 accumulated in the order x, y, z (vec3d::len)
        const double gg = g * g;
        g2 = dim == 0 ? gg : g2 + gg;
    }
    return (float)(sgn0 * (1.0 - sqrt(g2)));
}

// Euler: phi_out = fl(fl(d * dt) + phi) on the band
__global__ __launch_bounds__(256) void k_redist_euler(RShape s, Split sp, double dx, float dtf,
                                                      const uint32_t *__restrict__ list,
                                                      const unsigned int *__restrict__ count,
                                                      const float *__restrict__ phi, const float *__restrict__ phi0,
                                                      const float *__restrict__ sgn, const uint8_t *__restrict__ m,
                                                      float *__restrict__ phi_out) {
#pragma clang fp contract(off)
    const unsigned int len = *count;
    for (unsigned int e = blockIdx.x * 256 + threadIdx.x; e < len; e += gridDim.x * 256) {
        const uint32_t c = list[e];
        int i, j, k;
        decompose(c, sp, i, j, k);
        const float t = redist_rate(s, dx, phi, phi0, sgn, m, i, j, k, c) * dtf;
        phi_out[c] = t + phi[c];
    }
}

// RK2 first stage: d0 = rate(phi), tmp = fl(fl(d0 * dt) + phi) on the band
__global__ __launch_bounds__(256) void k_redist_rk_a(RShape s, Split sp, double dx, float dtf,
                                                     const uint32_t *__restrict__ list,
                                                     const unsigned int *__restrict__ count,
                                                     const float *__restrict__ phi, const float *__restrict__ phi0,
                                                     const float *__restrict__ sgn, const uint8_t *__restrict__ m,
                                                     float *__restrict__ d0, float *__restrict__ tmp) {
#pragma clang fp contract(off)
    const unsigned int len = *count;
    for (unsigned int e = blockIdx.x * 256 + threadIdx.x; e < len; e += gridDim.x * 256) {
        const uint32_t c = list[e];
        int i, j, k;
        decompose(c, sp, i, j, k);
        const float d = redist_rate(s, dx, phi, phi0, sgn, m, i, j, k, c);
        const float t = d * dtf;
        d0[c] = d;
        tmp[c] = t + phi[c];
    }
}

// RK2 second stage: phi_out = fl(phi + fl(fl(d0 + rate(tmp)) * fl(dt / 2)))
__global__ __launch_bounds__(256) void k_redist_rk_b(RShape s, Split sp, double dx, float hdtf,
                                                     const uint32_t *__restrict__ list,
                                                     const unsigned int *__restrict__ count,
                                                     const float *__restrict__ phi, const float *__restrict__ tmp,
                                                     const float *__restrict__ phi0, const float *__restrict__ sgn,
                                                     const uint8_t *__restrict__ m, const float *__restrict__ d0,
                                                     float *__restrict__ phi_out) {
#pragma clang fp contract(off)
    const unsigned int len = *count;
    for (unsigned int e = blockIdx.x * 256 + threadIdx.x; e < len; e += gridDim.x * 256) {
        const uint32_t c = list[e];
        int i, j, k;
        decompose(c, sp, i, j, k);
        const float d1 = redist_rate(s, dx, tmp, phi0, sgn, m, i, j, k, c);
        const float sum = d0[c] + d1;
        const float t = sum * hdtf;
        phi_out[c] = phi[c] + t;
    }
}

// The band cut at bw and the fill off it, four cells per thread; src holds the band's
// evolved values.  Only what changes is written: off the band most cells hold their fill.
__global__ __launch_bounds__(256) void k_redist_finish(int64_t n, double bw, const float *src,
                                                       const uint8_t *__restrict__ m, int vec, float *phi,
                                                       uint8_t *band, unsigned int *__restrict__ count) {
#pragma clang fp contract(off)
    unsigned int act = 0;
    const int64_t groups = (n + 3) / 4;
    for (int64_t g = blockIdx.x * (int64_t)256 + threadIdx.x; g < groups; g += (int64_t)gridDim.x * 256) {
        const int64_t c0 = 4 * g;
        const uchar4 tv = *reinterpret_cast<const uchar4 *>(m + c0);
        const uint8_t t[4] = {tv.x, tv.y, tv.z, tv.w};
        const bool whole = vec && c0 + 4 <= n;
        float f[4];
        uint8_t o[4];
        if (whole) {
            const float4 fv = *reinterpret_cast<const float4 *>(phi + c0);
            const uchar4 ov = *reinterpret_cast<const uchar4 *>(band + c0);
            f[0] = fv.x, f[1] = fv.y, f[2] = fv.z, f[3] = fv.w;
            o[0] = ov.x, o[1] = ov.y, o[2] = ov.z, o[3] = ov.w;
        } else {
            for (int q = 0; q < 4; ++q) {
                f[q] = c0 + q < n ? phi[c0 + q] : 0.0f;
                o[q] = c0 + q < n ? band[c0 + q] : 0;
            }
        }
        float v[4];
        uint8_t b[4];
        bool changed = false, moved = false;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = t[q] && c0 + q < n ? src[c0 + q] : f[q];
            b[q] = t[q] && !(fabs((double)v[q]) > bw) ? 1 : 0;
            if (!b[q]) v[q] = v[q] < 0.0f ? (float)(-bw) : (float)bw;
            if (c0 + q < n) act += b[q];
            changed = changed || __float_as_uint(v[q]) != __float_as_uint(f[q]);
            moved = moved || b[q] != o[q];
        }
        if (whole) {
            if (changed) *reinterpret_cast<float4 *>(phi + c0) = make_float4(v[0], v[1], v[2], v[3]);
            if (moved) *reinterpret_cast<uchar4 *>(band + c0) = make_uchar4(b[0], b[1], b[2], b[3]);
        } else {
            for (int q = 0; q < 4; ++q)
                if (c0 + q < n) {
                    phi[c0 + q] = v[q];
                    band[c0 + q] = b[q];
                }
        }
    }
    act = block_count(act);
    if (threadIdx.x == 0 && act) atomicAdd(count, act);
}

}  // namespace

}  // namespace shk

using namespace shk;

extern "C" int shk_redistance(shk_ctx *c, float *phi, uint8_t *band, int width, int64_t *active) {
    if (!c) return SHK_BAD_ARG;
    c->err.clear();
    if (!phi || !band) return c->fail(SHK_BAD_ARG, "NULL level set or band pointer");
    if (width < 1 || width > 64) return c->fail(SHK_BAD_ARG, "width must be in 1..64");
    if (c->dims.bx != 8) return c->fail(SHK_BAD_ARG, "shk_redistance needs a 3D context");
    if (c->prm.host_pointers) return c->fail(SHK_BAD_ARG, "shk_redistance takes device pointers");
    HIPC(c, hipSetDevice(c->device));
    const RShape s{c->dims.nx, c->dims.ny, c->dims.nz};
    const int64_t n = (int64_t)s.nx * s.ny * s.nz;
    if (!c->redist) c->redist = new RedistWork();
    RedistWork *w = c->redist;
    HIPC(c, w->m.ensure((size_t)(n + 3) / 4 * 4));
    HIPC(c, w->list.ensure(n));
    HIPC(c, w->p.ensure(n));
    HIPC(c, w->phi0.ensure(n));
    HIPC(c, w->sgn.ensure(n));
    HIPC(c, w->count.ensure(2));
    const bool rk2 = c->prm.redist_rk2;
    if (rk2) {
        HIPC(c, w->d0.ensure(n));
        HIPC(c, w->tmp.ensure(n));
    }
    hipStream_t st = c->stream;
    const Split sp{div32(s.nx), div32(s.ny)};
    const unsigned g4 = (unsigned)(((n + 3) / 4 + 255) / 256);
    const unsigned gl = (unsigned)std::min<int64_t>(kBandBlocks, (n + 255) / 256);
    const int vec_phi = (uintptr_t)phi % 16 == 0, vec_band = (uintptr_t)band % 4 == 0;
    const double dx = c->dx, rate = c->prm.redist_rate;
    unsigned int *len = w->count.p, *cnt_d = w->count.p + 1;
    const uint8_t *m = w->m.p;
    hipLaunchKernelGGL(k_zero_counts, dim3(1), dim3(64), 0, st, w->count.p, 2);
    hipLaunchKernelGGL(k_redist_trim, dim3(g4), dim3(256), 0, st, s, sp, phi, band, vec_band, w->m.p);
    for (int r = 1; r <= width; ++r)
        hipLaunchKernelGGL(k_redist_dilate, dim3(g4), dim3(256), 0, st, s, sp, r, s.nx % 4 == 0 ? 1 : 0, w->m.p);
    hipLaunchKernelGGL(k_band_list, dim3(band_list_blocks(n)), dim3(kBandNT), 0, st, n, m, 1, 0, w->list.p, len);
    hipLaunchKernelGGL(k_redist_init, dim3(gl), dim3(256), 0, st, dx, w->list.p, len, m, phi, w->phi0.p, w->sgn.p);
    // the steps alternate between the caller's array and the work array
    float *P[2] = {phi, w->p.p};
    int cur = 0;
    const float dtf = (float)(rate * dx), hdtf = (float)(0.5 * (rate * dx));
    const int iters = (int)std::ceil((double)width / rate);
    for (int it = 0; it < iters; ++it) {
        if (!rk2) {
            hipLaunchKernelGGL(k_redist_euler, dim3(gl), dim3(256), 0, st, s, sp, dx, dtf, w->list.p, len, P[cur],
                               w->phi0.p, w->sgn.p, m, P[cur ^ 1]);
        } else {
            hipLaunchKernelGGL(k_redist_rk_a, dim3(gl), dim3(256), 0, st, s, sp, dx, dtf, w->list.p, len, P[cur],
                               w->phi0.p, w->sgn.p, m, w->d0.p, w->tmp.p);
            hipLaunchKernelGGL(k_redist_rk_b, dim3(gl), dim3(256), 0, st, s, sp, dx, hdtf, w->list.p, len, P[cur],
                               w->tmp.p, w->phi0.p, w->sgn.p, m, w->d0.p, P[cur ^ 1]);
        }
        cur ^= 1;
    }
    hipLaunchKernelGGL(k_redist_finish, dim3(std::min(g4, kBandBlocks)), dim3(256), 0, st, n, dx * (double)width,
                       P[cur], m, vec_phi && vec_band, phi, band, cnt_d);
    HIPC(c, hipGetLastError());
    unsigned int cnt = 0;
    HIPC(c, hipMemcpyAsync(&cnt, cnt_d, sizeof cnt, hipMemcpyDeviceToHost, st));
    HIPC(c, hipStreamSynchronize(st));
    if (active) *active = (int64_t)cnt;
    return SHK_OK;
}
