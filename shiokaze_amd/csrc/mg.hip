// mg.hip -- aggregation multigrid V-cycle kernels on the brick layout (see mg.h).
//
// Every kernel returns when the Krylov state it is given has stopped, before it reads a
// vector, so the V-cycles queued behind a converged iteration cost little more than their
// launches; the brick tables are read before the state, so that the loads overlap.
#include "mg.h"

namespace shk {

namespace {

constexpr int NT = 256;

inline unsigned blocks(int64_t n) { return (unsigned)((n + NT - 1) / NT > 0 ? (n + NT - 1) / NT : 1); }

__device__ inline bool stopped(const SolveState *s) { return s && s->done; }

// uniform coupling of the brick (level 0), 0 when none
__device__ inline float brick_kappa(const MgOp &op, int slot) { return op.kappa ? op.kappa[slot] : 0.0f; }

// diagonal of cell e: 1 in a uniform brick
__device__ inline float diag_of(const MgOp &op, int64_t e, float kap) { return kap != 0.0f ? 1.0f : op.d[e]; }

// (A v)_e for the 7-point brick operator of a level >= 1 (explicit diagonal and
// couplings, FP32), where v(s, m) is the value at local cell m of slot s; a missing
// neighbour brick adds nothing.  A 2D grid (Y == 1) has no y neighbours.
template <int BX, class V>
__device__ inline float apply_v(const MgOp &op, int slot, int l, V v) {
    using B = BrickShape<BX>;
    constexpr int X = B::X, Y = B::Y;
    const int64_t e = (int64_t)slot * kBrickCells + l;
    const int i = l % X, j = (l / X) % Y, k = l / kWave;
    const int *nb = op.nbr + 6 * slot;
    float acc = op.d[e] * v(slot, l);
    if (i > 0) {
        acc -= op.cx[e] * v(slot, l - 1);
    } else if (nb[0] >= 0) {
        acc -= op.cx[e] * v(nb[0], l + (X - 1));
    }
    if (i < X - 1) {
        acc -= op.cx[e + 1] * v(slot, l + 1);
    } else if (nb[1] >= 0) {
        acc -= op.cx[(int64_t)nb[1] * kBrickCells + l - (X - 1)] * v(nb[1], l - (X - 1));
    }
    if constexpr (Y > 1) {
        if (j > 0) {
            acc -= op.cy[e] * v(slot, l - X);
        } else if (nb[2] >= 0) {
            acc -= op.cy[e] * v(nb[2], l + X * (Y - 1));
        }
        if (j < Y - 1) {
            acc -= op.cy[e + X] * v(slot, l + X);
        } else if (nb[3] >= 0) {
            acc -= op.cy[(int64_t)nb[3] * kBrickCells + l - X * (Y - 1)] * v(nb[3], l - X * (Y - 1));
        }
    }
    if (k > 0) {
        acc -= op.cz[e] * v(slot, l - 64);
    } else if (nb[4] >= 0) {
        acc -= op.cz[e] * v(nb[4], l + 448);
    }
    if (k < 7) {
        acc -= op.cz[e + 64] * v(slot, l + 64);
    } else if (nb[5] >= 0) {
        acc -= op.cz[(int64_t)nb[5] * kBrickCells + l - 448] * v(nb[5], l - 448);
    }
    return acc;
}

// Aggregation: 2x2x2 children per coarse cell, 2x1x2 on a 2D grid (Y == 1).
template <int BX>
struct Agg {
    using B = BrickShape<BX>;
    static constexpr int X = B::X, Y = B::Y;
    static constexpr int AY = Y > 1 ? 2 : 1;       // aggregation factor along y
    static constexpr int NCH = 4 * AY;             // children per coarse cell
    // brick-local offset of child q (a along x, b along y, c along z)
    __device__ static int child(int q) {
        const int a = q & 1, b = AY > 1 ? (q >> 1) & 1 : 0, c = AY > 1 ? q >> 2 : q >> 1;
        return a + X * b + 64 * c;
    }
    __device__ static void bits(int q, int &a, int &b, int &c) {
        a = q & 1;
        b = AY > 1 ? (q >> 1) & 1 : 0;
        c = AY > 1 ? q >> 2 : q >> 1;
    }
};

// fine slot holding the children of coarse cell (slot_c, l) and the children's base
// local offset; -1 when the fine brick is outside the grid or inactive
template <int BX>
__device__ inline int children(const MgLevelDev &f, const MgLevelDev &c, int slot_c, int l, int &base) {
    using A = Agg<BX>;
    constexpr int X = A::X, Y = A::Y, HX = X / 2, HY = Y > 1 ? Y / 2 : 1;
    const int ci = l % X, cj = (l / X) % Y, ck = l / kWave;
    const int4 Bc = c.coord[slot_c];
    if (Bc.x * X + ci >= c.nx || Bc.y * Y + cj >= c.ny || Bc.z * 8 + ck >= c.nz) return -1;
    const int fbx = 2 * Bc.x + ci / HX, fby = A::AY * Bc.y + cj / HY, fbz = 2 * Bc.z + (ck >> 2);
    if (fbx >= f.nbx || fby >= f.nby || fbz >= f.nbz) return -1;
    base = 2 * (ci % HX) + X * (A::AY * (cj % HY)) + 64 * (2 * (ck & 3));
    return f.slot[fbx + f.nbx * (fby + f.nby * fbz)];
}

// cell index on the next level of the cell (brick coord Bf, local l) of a fine level
template <int BX>
__device__ inline int coarse_local(int4 Bf, int l) {
    using A = Agg<BX>;
    constexpr int X = A::X, Y = A::Y, HX = X / 2, HY = Y > 1 ? Y / 2 : 1;
    const int i = l % X, j = (l / X) % Y, k = l / kWave;
    const int cy = A::AY > 1 ? (Bf.y & 1) * HY + j / 2 : 0;
    return ((Bf.x & 1) * HX + i / 2) + X * cy + 64 * ((Bf.z & 1) * 4 + k / 2);
}

__global__ __launch_bounds__(NT) void k_mg_mask(int64_t n, const double *__restrict__ sig, float *__restrict__ d0) {
    const int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x;
    if (e < n) d0[e] = sig[e] > 0.0 ? 1.0f : 0.0f;
}

template <int BX>
__global__ __launch_bounds__(NT) void k_mg_coarsen(MgLevelDev f, MgLevelDev c, float4 *__restrict__ dense,
                                                  int sx, int sxy) {
    using A = Agg<BX>;
    const int64_t E = blockIdx.x * (int64_t)NT + threadIdx.x;
    if (E >= (int64_t)c.n_active * kBrickCells) return;
    const int slot_c = (int)(E >> 9), l = (int)(E & 511);
    int base = 0;
    const int fs = children<BX>(f, c, slot_c, l, base);
    double d = 0.0, inner = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
    if (fs >= 0) {
        const int64_t fb = (int64_t)fs * kBrickCells + base;
#pragma unroll
        for (int q = 0; q < A::NCH; ++q) {
            int a, b, cc;
            A::bits(q, a, b, cc);
            const int64_t e = fb + A::child(q);
            d += (double)f.d[e];
            if (a) inner += (double)f.cx[e]; else cx += (double)f.cx[e];
            if (A::AY > 1) {
                if (b) inner += (double)f.cy[e]; else cy += (double)f.cy[e];
            }
            if (cc) inner += (double)f.cz[e]; else cz += (double)f.cz[e];
        }
    }
    double dc = d - 2.0 * inner;
    if (!(dc > 1e-6 * d)) dc = 0.0;  // no unknown child, or an aggregate decoupled from every boundary
    c.d[E] = (float)dc;
    c.cx[E] = (float)cx;
    c.cy[E] = (float)cy;
    c.cz[E] = (float)cz;
    if (dense) {
        constexpr int X = A::X, Y = A::Y;
        const int4 B = c.coord[slot_c];
        const int i = B.x * X + l % X, j = B.y * Y + (l / X) % Y, k = B.z * 8 + l / kWave;
        if (i < c.nx && j < c.ny && k < c.nz)
            dense[i + sx * j + sxy * k] = make_float4((float)dc, (float)cx, (float)cy, (float)cz);
    }
    // k_mg_residual_restrict does not write the cells without a fine brick
    c.b[E] = 0.0f;
    c.x[E] = 0.0f;
}

// b_c = P0' (b_f - A_f x_f), x_c = w b_c / d_c (0 with w = 0) from a level >= 1, one
// thread per fine cell: each cell's residual goes to LDS and is never stored; the
// first child of each aggregate sums its children in the order q (the children of an
// aggregate lie in one 256-cell half brick, the z pairs (2m, 2m+1) never straddle
// the halves).  Coarse cells without a fine brick are not written: their b and x
// hold the zeros k_mg_coarsen writes, and nothing else writes there.
template <int BX>
__global__ __launch_bounds__(NT) void k_mg_residual_restrict(MgLevelDev f, MgLevelDev c, float omega,
                                                             const SolveState *state) {
    using A = Agg<BX>;
    constexpr int X = A::X, Y = A::Y;
    static_assert(kBrickCells % NT == 0 && NT % (2 * kWave) == 0, "a block holds whole z pairs of one brick");
    __shared__ float ts[NT];
    const int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x;
    if (e >= (int64_t)f.n_active * kBrickCells) return;  // whole blocks: n_active * 512 is a multiple of NT
    const int slot = (int)(e >> 9), l = (int)(e & 511);
    // every load is issued before the barrier, none waits on the residual: the parent
    // cell's diagonal, then the residual's operands (all in bounds whatever d is)
    const int ps = f.parent[slot];  // >= 0: the parent of an active brick is active
    const int64_t E = (int64_t)(ps > 0 ? ps : 0) * kBrickCells + coarse_local<BX>(f.coord[slot], l);
    if (stopped(state)) return;
    const float dc = c.d[E];
    const MgOp op = f.op(0.0f, 0.0f);
    const float *__restrict__ xf = f.x;
    const auto v = [xf](int sl, int m) { return xf[(int64_t)sl * kBrickCells + m]; };
    const float ax = apply_v<BX>(op, slot, l, v);
    ts[threadIdx.x] = f.d[e] > 0.0f ? f.b[e] - ax : 0.0f;
    __syncthreads();
    const int i = l % X, j = (l / X) % Y, k = l / kWave;
    if ((i & 1) || (A::AY > 1 && (j & 1)) || (k & 1) || ps < 0) return;
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < A::NCH; ++q) s += ts[threadIdx.x + A::child(q)];
    c.b[E] = dc > 0.0f ? s : 0.0f;
    c.x[E] = dc > 0.0f ? omega * s / dc : 0.0f;
}

// x_f += alpha P0 x_c on the unknowns of a level f >= 1, one thread per cell (the
// level above the tail; the others get theirs from k_mg_smooth)
template <int BX>
__global__ __launch_bounds__(NT) void k_mg_prolong(MgLevelDev f, MgLevelDev c, float alpha, const SolveState *state) {
    const int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x;
    if (e >= (int64_t)f.n_active * kBrickCells) return;
    const int slot = (int)(e >> 9), l = (int)(e & 511);
    const int ps = f.parent[slot];  // >= 0: the parent of an active brick is active
    const int64_t E = (int64_t)(ps > 0 ? ps : 0) * kBrickCells + coarse_local<BX>(f.coord[slot], l);
    if (stopped(state)) return;
    const float dv = f.d[e], xe = f.x[e], xc = c.x[E];
    if (dv > 0.0f && ps >= 0) f.x[e] = fmaf(alpha, xc, xe);
}

// c.t = y = x + w (b - A x) / d on a level >= 1, one thread per cell; with a finer
// level f >= 1 (prolong) the same thread also adds alpha y to the unknowns among its
// children there (f.x += alpha P0 y, the next coarse correction, which k_mg_prolong
// would make from the stored y)
template <int BX>
__global__ __launch_bounds__(NT) void k_mg_smooth(MgLevelDev c, MgLevelDev f, bool prolong, float omega, float alpha,
                                                  const SolveState *state) {
    using A = Agg<BX>;
    const int64_t e = blockIdx.x * (int64_t)NT + threadIdx.x;
    if (e >= (int64_t)c.n_active * kBrickCells) return;
    const int slot = (int)(e >> 9), l = (int)(e & 511);
    // the children's d and x are loaded with the smoothing's operands, not after them
    int base = 0;
    const int fs = prolong ? children<BX>(f, c, slot, l, base) : -1;
    if (stopped(state)) return;
    const int64_t fb = (int64_t)(fs > 0 ? fs : 0) * kBrickCells + base;
    float fd[A::NCH], fx[A::NCH];
#pragma unroll
    for (int q = 0; q < A::NCH; ++q) {
        fd[q] = fs >= 0 ? f.d[fb + A::child(q)] : 0.0f;
        fx[q] = fs >= 0 ? f.x[fb + A::child(q)] : 0.0f;
    }
    const MgOp op = c.op(omega, alpha);
    const float *__restrict__ x = c.x;
    const auto v = [x](int sl, int m) { return x[(int64_t)sl * kBrickCells + m]; };
    const float dv = c.d[e], xe = x[e], be = c.b[e];
    const float ax = apply_v<BX>(op, slot, l, v);  // all loads in bounds whatever d is
    const float y = dv > 0.0f ? xe + omega * (be - ax) / dv : 0.0f;
    c.t[e] = y;
#pragma unroll
    for (int q = 0; q < A::NCH; ++q)
        if (fd[q] > 0.0f) f.x[fb + A::child(q)] = fmaf(alpha, y, fx[q]);  // one rounding, as k_mg_prolong
}

// ---- level 0, fused.  On the scaled system every level-0 vector is zero off the
// unknowns and the diagonal is 1 on them, so x0 = w r needs no division and is never
// stored: the pre-smoothing residual and the post-smoothing recompute it from r.

// value of x0' = w r + alpha P0 x1 at level-0 cell (slot, l) of brick B with parent ps
template <int BX>
__device__ inline float xprime(const MgOp &op, const float *__restrict__ r, const float *__restrict__ xc, int slot,
                               int l, int4 B, int ps) {
    return op.omega * r[(int64_t)slot * kBrickCells + l] +
           op.alpha * xc[(int64_t)ps * kBrickCells + coarse_local<BX>(B, l)];
}

// ---------------------------------------------------------------- level 0, one wave per brick
//
// The two level-0 passes with PL z-planes of a brick per wave: lane = i + X j holds one
// (x, y) column (X x Y = 64: 8 x 8 for 3D bricks, 64 x 1 for the 64x1x8 bricks of 2D grids)
// of the planes.  PL = 8, the whole brick, reads least; PL = 2 puts four times the waves on
// the chip and quarters each one's chain of shuffles, which is what bounds a small grid
// (kMgSplitBricks).  In-brick x and y neighbours come by lane
// shuffles (taken by all 64 lanes, outside any lane-dependent branch), z neighbours
// from the lane's own registers, and the cells across the faces from one coalesced
// load per neighbour plane (the neighbour brick's slot, coordinates and parent are
// wave-uniform).  Each cell's arithmetic takes its terms in the face order of
// apply_v<BX> (-x, +x, -y, +y, -z, +z); a uniform brick sums its six neighbours
// first and scales the sum by its one coupling.

__device__ inline float lane_get(float v, int src) { return __shfl(v, src & 63, 64); }

// the cells across the faces of a brick as plane registers (0 where the neighbour
// brick does not exist): x planes hold (y = a, z = c) at lane a + Y c (the first 8 Y
// lanes), y planes (x = a, z = c) at lane a + X c, z planes (x, y) at the lane itself
template <int BX, class V>
__device__ inline void halo_planes(const int nb[6], int lane, V value, float h[6]) {
    using B = BrickShape<BX>;
    constexpr int X = B::X, Y = B::Y;
    const int xa = lane % Y, xc = lane / Y;
    const bool xl = lane < Y * 8;
    h[0] = nb[0] >= 0 && xl ? value(nb[0], (X - 1) + X * xa + 64 * xc) : 0.0f;
    h[1] = nb[1] >= 0 && xl ? value(nb[1], X * xa + 64 * xc) : 0.0f;
    h[2] = h[3] = 0.0f;
    if constexpr (Y > 1) {
        const int pa = lane % X, pc = lane / X;
        h[2] = nb[2] >= 0 ? value(nb[2], pa + X * (Y - 1) + 64 * pc) : 0.0f;
        h[3] = nb[3] >= 0 ? value(nb[3], pa + 64 * pc) : 0.0f;
    }
    h[4] = nb[4] >= 0 ? value(nb[4], lane + 448) : 0.0f;
    h[5] = nb[5] >= 0 ? value(nb[5], lane) : 0.0f;
}

// the six neighbour values of cell (i, j, k) in face order x-, x+, y-, y+, z-, z+
// (y values 0 without a y axis); v: the wave's planes k0 .. k0 + PL - 1, zl and zh those
// around them
template <int BX, int PL>
__device__ inline void neighbours6(const float *v, const float h[6], float zl, float zh, int lane, int k0, int p,
                                   float n[6]) {
    using B = BrickShape<BX>;
    constexpr int X = B::X, Y = B::Y;
    const int i = lane % X, j = lane / X, k = k0 + p;
    const float x0 = v[p];
    float xm = lane_get(x0, lane - 1), xp = lane_get(x0, lane + 1);
    const float hxm = lane_get(h[0], j + Y * k), hxp = lane_get(h[1], j + Y * k);
    if (i == 0) xm = hxm;
    if (i == X - 1) xp = hxp;
    float ym = 0.0f, yp = 0.0f;
    if constexpr (Y > 1) {
        ym = lane_get(x0, lane - X);
        yp = lane_get(x0, lane + X);
        const float hym = lane_get(h[2], i + X * k), hyp = lane_get(h[3], i + X * k);
        if (j == 0) ym = hym;
        if (j == Y - 1) yp = hyp;
    }
    n[0] = xm;
    n[1] = xp;
    n[2] = ym;
    n[3] = yp;
    n[4] = p > 0 ? v[p > 0 ? p - 1 : 0] : zl;
    n[5] = p < PL - 1 ? v[p < PL - 1 ? p + 1 : p] : zh;
}

// the couplings of cell e across its faces (low faces live at e, high faces at the
// neighbour cell) and whether each neighbour exists; a uniform brick has kap on all
template <int BX>
__device__ inline void couplings6(const MgOp &op, int64_t e, const int nb[6], int lane, int k, float kap, float c[6],
                                  bool has[6]) {
    using B = BrickShape<BX>;
    constexpr int X = B::X, Y = B::Y;
    const int i = lane % X, j = lane / X;
    has[0] = i > 0 || nb[0] >= 0;
    has[1] = i < X - 1 || nb[1] >= 0;
    has[2] = Y > 1 && (j > 0 || nb[2] >= 0);
    has[3] = Y > 1 && (j < Y - 1 || nb[3] >= 0);
    has[4] = k > 0 || nb[4] >= 0;
    has[5] = k < 7 || nb[5] >= 0;
    if (kap != 0.0f) {
#pragma unroll
        for (int f = 0; f < 6; ++f) c[f] = kap;
        return;
    }
    c[0] = op.cx[e];
    c[1] = i < X - 1 ? op.cx[e + 1]
                     : (nb[1] >= 0 ? op.cx[(int64_t)nb[1] * kBrickCells + lane - (X - 1) + 64 * k] : 0.0f);
    c[2] = c[3] = 0.0f;
    if constexpr (Y > 1) {
        c[2] = op.cy[e];
        c[3] = j < Y - 1 ? op.cy[e + X]
                         : (nb[3] >= 0 ? op.cy[(int64_t)nb[3] * kBrickCells + lane - X * (Y - 1) + 64 * k] : 0.0f);
    }
    c[4] = op.cz[e];
    c[5] = k < 7 ? op.cz[e + 64] : (nb[5] >= 0 ? op.cz[(int64_t)nb[5] * kBrickCells + lane] : 0.0f);
}

// the brick and the first plane of this wave
template <int PL>
__device__ inline int wave_brick(int &k0) {
    const int w = blockIdx.x * (NT / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    k0 = PL * (w % (8 / PL));
    return w / (8 / PL);
}

// t0 = r - A (w r) = r - w A r on the unknowns (0 elsewhere), by linearity, restricted
// at once to level 1 (b_1 = P0' t0, x_1 = w_c b_1 / d_1)
template <int BX, int PL>
__global__ __launch_bounds__(NT) void k_mg_pre0_w(MgOp op, const float *__restrict__ r, const int4 *__restrict__ coord,
                                                  const int *__restrict__ parent, MgLevelDev c, float omega_c,
                                                  const SolveState *state) {
    constexpr int X = BrickShape<BX>::X, Y = BrickShape<BX>::Y;
    const int lane = threadIdx.x & 63;
    int k0;
    const int slot = wave_brick<PL>(k0);
    if (slot >= op.n_active) return;   // no block-wide synchronisation below
    int nb[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) nb[f] = op.nbr[6 * slot + f];
    const float kap = brick_kappa(op, slot);
    const int64_t base = (int64_t)slot * kBrickCells + lane;
    const int ps = parent[slot];  // >= 0: the parent of an active brick is active
    const int4 Bf = coord[slot];
    if (stopped(state)) return;
    float dcm[PL / 2];  // level-1 diagonals of the cells this lane may restrict to, loaded early
#pragma unroll
    for (int m = 0; m < PL / 2; ++m)
        dcm[m] = c.d[(int64_t)(ps > 0 ? ps : 0) * kBrickCells + coarse_local<BX>(Bf, lane + 64 * (k0 + 2 * m))];
    const auto value = [&](int ns, int l) { return r[(int64_t)ns * kBrickCells + l]; };
    float v[PL];
#pragma unroll
    for (int p = 0; p < PL; ++p) v[p] = r[base + 64 * (k0 + p)];
    float h[6];
    halo_planes<BX>(nb, lane, value, h);
    const float zl = k0 > 0 ? value(slot, lane + 64 * (k0 - 1)) : h[4];
    const float zh = k0 + PL < 8 ? value(slot, lane + 64 * (k0 + PL)) : h[5];
    float t[PL];
#pragma unroll
    for (int p = 0; p < PL; ++p) {
        const int64_t e = base + 64 * (k0 + p);
        float n[6];
        neighbours6<BX, PL>(v, h, zl, zh, lane, k0, p, n);
        float ax;
        if (kap != 0.0f) {
            // the y terms are 0.0f without a y axis
            ax = v[p] - kap * (n[0] + n[1] + (Y > 1 ? n[2] : 0.0f) + (Y > 1 ? n[3] : 0.0f) + n[4] + n[5]);
        } else {
            float c[6];
            bool has[6];
            couplings6<BX>(op, e, nb, lane, k0 + p, kap, c, has);
            ax = op.d[e] * v[p];
#pragma unroll
            for (int f = 0; f < 6; ++f)
                if (has[f]) ax -= c[f] * n[f];
        }
        t[p] = diag_of(op, e, kap) > 0.0f ? v[p] - op.omega * ax : 0.0f;
    }
    // b_1 = P0' t and x_1 = w_c b_1 / d_1 on the coarse cells whose children are in
    // this brick: a cell of even (i, j, k) sums the children (i+a, j+b, k+c) in the
    // order a, b, c (that of Agg<BX>::child), taken from lanes +1, +X, +X+1 and its
    // own next register; t is not stored
    float sum[PL / 2];
#pragma unroll
    for (int m = 0; m < PL / 2; ++m) {
        float q[8];
#pragma unroll
        for (int cz = 0; cz < 2; ++cz) {
            const float tv = t[2 * m + cz];
            q[4 * cz] = tv;
            q[4 * cz + 1] = lane_get(tv, lane + 1);
            q[4 * cz + 2] = Y > 1 ? lane_get(tv, lane + X) : 0.0f;
            q[4 * cz + 3] = Y > 1 ? lane_get(tv, lane + X + 1) : 0.0f;
        }
        float sm = 0.0f;
#pragma unroll
        for (int cz = 0; cz < 2; ++cz) {
            sm += q[4 * cz];
            sm += q[4 * cz + 1];
            if constexpr (Y > 1) {
                sm += q[4 * cz + 2];
                sm += q[4 * cz + 3];
            }
        }
        sum[m] = sm;
    }
    const int i = lane % X, j = lane / X;
    if ((i & 1) || (Y > 1 && (j & 1)) || ps < 0) return;  // ps < 0 cannot happen for an active brick
#pragma unroll
    for (int m = 0; m < PL / 2; ++m) {
        const int64_t E = (int64_t)ps * kBrickCells + coarse_local<BX>(Bf, lane + 64 * (k0 + 2 * m));
        const float dc = dcm[m];
        c.b[E] = dc > 0.0f ? sum[m] : 0.0f;
        c.x[E] = dc > 0.0f ? omega_c * sum[m] / dc : 0.0f;
    }
}

// y = x0' + w (r - A x0') with x0' = w r + alpha P0 x1 computed on the fly (the
// prolongation fused into the post-smoothing); part[block] = sum r*y over the block's
// planes
template <int BX, int PL>
__global__ __launch_bounds__(NT) void k_mg_post0_w(MgOp op, const int4 *__restrict__ coord,
                                                   const int *__restrict__ parent, const float *__restrict__ r,
                                                   const float *__restrict__ xc, float *__restrict__ y,
                                                   const SolveState *state, double *__restrict__ part) {
    __shared__ double lds[NT / kWave];
    const int lane = threadIdx.x & 63;
    int k0;
    const int slot = wave_brick<PL>(k0);
    const int sl = slot < op.n_active ? slot : 0;
    double acc = 0.0;
    int nb[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) nb[f] = op.nbr[6 * sl + f];
    const float kap = brick_kappa(op, sl);
    const int4 B = coord[sl];
    const int ps = parent[sl];
    if (stopped(state)) return;
    if (slot < op.n_active) {
        const int64_t base = (int64_t)slot * kBrickCells + lane;
        const auto own = [&](int k) { return xprime<BX>(op, r, xc, slot, lane + 64 * k, B, ps); };
        float rv[PL], xs[PL];
#pragma unroll
        for (int p = 0; p < PL; ++p) {
            rv[p] = r[base + 64 * (k0 + p)];
            xs[p] = own(k0 + p);
        }
        float h[6];
        halo_planes<BX>(nb, lane,
                        [&](int ns, int l) { return xprime<BX>(op, r, xc, ns, l, coord[ns], parent[ns]); }, h);
        const float zl = k0 > 0 ? own(k0 - 1) : h[4], zh = k0 + PL < 8 ? own(k0 + PL) : h[5];
#pragma unroll
        for (int p = 0; p < PL; ++p) {
            const int64_t e = base + 64 * (k0 + p);
            float yv = 0.0f;
            // every lane takes part in the shuffles, whether its cell is an unknown or not
            float n[6];
            neighbours6<BX, PL>(xs, h, zl, zh, lane, k0, p, n);
            if (diag_of(op, e, kap) > 0.0f) {
                float c[6];
                bool has[6];
                couplings6<BX>(op, e, nb, lane, k0 + p, kap, c, has);
                float sum = 0.0f;
#pragma unroll
                for (int f = 0; f < 6; ++f)
                    if (has[f] && c[f] != 0.0f) sum += c[f] * n[f];
                yv = xs[p] + op.omega * (rv[p] - (xs[p] - sum));
            }
            y[e] = yv;
            acc += (double)rv[p] * (double)yv;
        }
    }
    const double s = block_sum<NT>(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// out[t] = sum of in[t*per .. (t+1)*per) for t < n_out, in a fixed order (the
// per-block partials of k_mg_post0_w, where the Krylov kernels should not fold them all)
__global__ __launch_bounds__(NT) void k_mg_fold(int n_in, const double *__restrict__ in, int n_out,
                                                double *__restrict__ out, const SolveState *state) {
    if (stopped(state)) return;
    const int t = blockIdx.x * NT + threadIdx.x;
    if (t >= n_out) return;
    const int per = (n_in + n_out - 1) / n_out;
    double s = 0.0;
    for (int q = t * per; q < (t + 1) * per && q < n_in; ++q) s += in[q];
    out[t] = s;
}

// The coarse end of the V-cycle -- the levels of T, down to the dense solve and back up --
// in one workgroup with the operators and vectors in LDS.  These levels hold too little work
// to fill the chip, so as one launch per pass they cost what a launch and its chain of
// dependent loads cost (4 to 5 us each); here a pass costs its LDS reads and a barrier.  One
// CU's instruction rate bounds it, so each level is a dense grid with a zero cell between
// rows, a zero row between planes and a zero plane between levels: a cell's neighbours are at
// fixed distances, with no edge tests (their zeros change no sum).  Every cell's arithmetic
// is that of the per-level kernels, term by term.  One V-cycle of 70x61x52 (tail of 18x16x13,
// 9x8x7, 5x4x4, 3x2x2): 13.1 us here instead of 27 in eight launches.
constexpr int TNT = 1024;
typedef float f4 __attribute__((ext_vector_type(4)));

struct TailLevel {
    int at, n, inner, nx, ny, cells, sx, sxy;   // first cell, size with and without the last zero plane
    float rx, ry;
    __device__ TailLevel(const MgTail &T, int t)
        : at(T.first[t]), n(T.first[t + 1] - T.first[t]), inner(T.sxy[t] * T.nz[t]), nx(T.nx[t]), ny(T.ny[t]),
          cells(T.nx[t] * T.ny[t] * T.nz[t]), sx(T.nx[t] + 1), sxy(T.sxy[t]), rx(1.0f / (float)T.nx[t]),
          ry(1.0f / (float)T.ny[t]) {}
    // cell c of nx x ny x nz, c < 2^13: (c + 0.5) / n is at least 0.5 / n away from a whole
    // number, far more than it rounds
    __device__ void split(int c, int &i, int &j, int &k) const {
        const int q = (int)(((float)c + 0.5f) * rx);
        i = c - q * nx;
        k = (int)(((float)q + 0.5f) * ry);
        j = q - k * ny;
    }
};

// A x at cell c (its operator in o): the terms of apply_v in its order
template <int BX>
__device__ inline float tail_apply(const f4 *__restrict__ op, const float *__restrict__ x, f4 o, int c, int sx,
                                   int sxy) {
    float acc = o.x * x[c];
    acc -= o.y * x[c - 1];
    acc -= op[c + 1].y * x[c + 1];
    if constexpr (BrickShape<BX>::Y > 1) {
        acc -= o.z * x[c - sx];
        acc -= op[c + sx].z * x[c + sx];
    }
    acc -= o.w * x[c - sxy];
    acc -= op[c + sxy].w * x[c + sxy];
    return acc;
}

template <int BX>
__global__ __launch_bounds__(TNT) void k_mg_tail(MgTail T, float omega, float alpha, const SolveState *state) {
    using A = Agg<BX>;
    constexpr int kPer = (kMgTailCells + TNT - 1) / TNT;
    __shared__ f4 op[kMgTailCells];   // d, cx, cy, cz
    // bt: b of the levels after the first (whose b stays in registers); the first level's
    // place holds the residuals of the level at work
    __shared__ float xs[kMgTailCells], bt[kMgTailCells];
    __shared__ int idx[kMgCoarseMax];
    static_assert(kMgCoarseMax == kWave, "one wave solves the coarsest level");
    const int tid = threadIdx.x, N = T.first[T.levels], nc = T.ncoarse;
    const TailLevel L0(T, 0);
    // one batch of loads for everything the cycle reads
    f4 ob[kPer];
    float xb[kPer], b0[kPer], iv[kMgCoarseMax];
    int src[kPer];
#pragma unroll
    for (int m = 0; m < kPer; ++m) src[m] = tid + TNT * m < L0.n ? T.src[tid + TNT * m] : -1;
    if (stopped(state)) return;
#pragma unroll
    for (int m = 0; m < kPer; ++m)
        if (tid + TNT * m < N) ob[m] = reinterpret_cast<const f4 *>(T.op)[tid + TNT * m];
    if (tid < nc) idx[tid] = T.idx[tid];
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
        xb[m] = src[m] >= 0 ? T.x[src[m]] : 0.0f;
        b0[m] = src[m] >= 0 ? T.b[src[m]] : 0.0f;
    }
#pragma unroll
    for (int m = 0; m < kPer; ++m)
        if (tid + TNT * m < N) {
            op[tid + TNT * m] = ob[m];
            xs[tid + TNT * m] = bt[tid + TNT * m] = 0.0f;
        }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kPer; ++m)
        if (src[m] >= 0) xs[L0.at + tid + TNT * m] = xb[m];
    if (T.levels == 1) {   // the coarsest alone: its b where the solve reads it
#pragma unroll
        for (int m = 0; m < kPer; ++m)
            if (src[m] >= 0) bt[L0.at + tid + TNT * m] = b0[m];
    }
    // the coarsest inverse, a row to each lane of the first wave
    if (tid < kMgCoarseMax)
#pragma unroll
        for (int j = 0; j < kMgCoarseMax; ++j) iv[j] = T.inv[j * kMgCoarseMax + tid];
    __syncthreads();
    float *const ts = bt + L0.at;
    for (int t = 0; t + 1 < T.levels; ++t) {
        const TailLevel F(T, t), C(T, t + 1);
#pragma unroll
        for (int m = 0; m < kPer; ++m) {
            const int l = tid + TNT * m, c = F.at + l;
            if (l >= F.n) break;
            float r = 0.0f;
            if (l < F.inner) {
                const f4 o = op[c];
                const float ax = tail_apply<BX>(op, xs, o, c, F.sx, F.sxy);
                r = o.x > 0.0f ? (t ? bt[c] : b0[m]) - ax : 0.0f;
            }
            ts[l] = r;
        }
        __syncthreads();
        const float w = t + 2 < T.levels ? omega : 0.0f;
        for (int l = tid; l < C.cells; l += TNT) {
            int i, j, k;
            C.split(l, i, j, k);
            const int c = C.at + i + (A::AY > 1 ? C.sx * j : 0) + C.sxy * k;
            const float *f = ts + 2 * i + (A::AY > 1 ? 2 * F.sx * j : 0) + 2 * F.sxy * k;
            float s = 0.0f;
#pragma unroll
            for (int q = 0; q < A::NCH; ++q) {
                int a, b, d;
                A::bits(q, a, b, d);
                s += f[a + F.sx * b + F.sxy * d];
            }
            const float dc = op[c].x;
            bt[c] = dc > 0.0f ? s : 0.0f;
            xs[c] = dc > 0.0f ? w * s / dc : 0.0f;
        }
        __syncthreads();
    }
    const int Z = T.first[T.levels - 1];
    if (tid < kMgCoarseMax) {
        const int at = Z + (tid < nc ? idx[tid] : 0);
        const float bv = tid < nc ? bt[at] : 0.0f;
        float acc = 0.0f;   // beyond nc both factors are zero
#pragma unroll
        for (int j = 0; j < kMgCoarseMax; ++j)
            acc += iv[j] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(bv), j));
        if (tid < nc) xs[at] = acc;   // the other cells of this level hold zeros
    }
    __syncthreads();
    for (int t = T.levels - 2; t >= 0; --t) {
        const TailLevel F(T, t), C(T, t + 1);
        for (int l = tid; l < C.cells; l += TNT) {
            int i, j, k;
            C.split(l, i, j, k);
            const float v = xs[C.at + i + (A::AY > 1 ? C.sx * j : 0) + C.sxy * k];
            const int f = F.at + 2 * i + (A::AY > 1 ? 2 * F.sx * j : 0) + 2 * F.sxy * k;
#pragma unroll
            for (int q = 0; q < A::NCH; ++q) {
                int a, b, d;
                A::bits(q, a, b, d);
                const int e = f + a + F.sx * b + F.sxy * d;
                if (op[e].x > 0.0f) xs[e] = fmaf(alpha, v, xs[e]);
            }
        }
        __syncthreads();
        float y[kPer];
#pragma unroll
        for (int m = 0; m < kPer; ++m) {
            const int l = tid + TNT * m, c = F.at + l;
            if (l >= F.inner) break;
            const f4 o = op[c];
            const float ax = tail_apply<BX>(op, xs, o, c, F.sx, F.sxy);
            y[m] = o.x > 0.0f ? xs[c] + omega * ((t ? bt[c] : b0[m]) - ax) / o.x : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < kPer; ++m)
            if (tid + TNT * m < F.inner) xs[F.at + tid + TNT * m] = y[m];
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < kPer; ++m)
        if (src[m] >= 0) T.x[src[m]] = xs[L0.at + tid + TNT * m];
}

}  // namespace

void launch_mg_mask(hipStream_t st, int64_t n, const double *sig, float *d0) {
    hipLaunchKernelGGL(k_mg_mask, dim3(blocks(n)), dim3(NT), 0, st, n, sig, d0);
}

#define SHK_MG_LAUNCH(kernel, bx, grid, ...)                                                   \
    do {                                                                                       \
        if ((bx) == 64)                                                                        \
            hipLaunchKernelGGL(kernel<64>, dim3(grid), dim3(NT), 0, __VA_ARGS__);              \
        else                                                                                   \
            hipLaunchKernelGGL(kernel<8>, dim3(grid), dim3(NT), 0, __VA_ARGS__);               \
    } while (0)

void launch_mg_coarsen(hipStream_t st, const MgLevelDev &f, const MgLevelDev &c, float4 *dense, int sx, int sxy) {
    SHK_MG_LAUNCH(k_mg_coarsen, c.bx, blocks((int64_t)c.n_active * kBrickCells), st, f, c, dense, sx,
                  sxy);
}

void launch_mg_residual_restrict(hipStream_t st, const MgLevelDev &f, const MgLevelDev &c, float omega,
                                 const SolveState *state) {
    SHK_MG_LAUNCH(k_mg_residual_restrict, f.bx, blocks((int64_t)f.n_active * kBrickCells), st, f, c, omega, state);
}

void launch_mg_prolong(hipStream_t st, const MgLevelDev &f, const MgLevelDev &c, float alpha, const SolveState *state) {
    SHK_MG_LAUNCH(k_mg_prolong, f.bx, blocks((int64_t)f.n_active * kBrickCells), st, f, c, alpha, state);
}

void launch_mg_smooth(hipStream_t st, const MgLevelDev &c, const MgLevelDev *fine, float omega, float alpha,
                      const SolveState *state) {
    const MgLevelDev none{};
    SHK_MG_LAUNCH(k_mg_smooth, c.bx, blocks((int64_t)c.n_active * kBrickCells), st, c, fine ? *fine : none,
                  fine != nullptr, omega, alpha, state);
}

// Level-0 grids of up to this many bricks are split four ways per brick, above it the chip is
// full and a wave keeps its brick.  One iteration, whole bricks / split: 70x61x52 (284 bricks)
// 72.5 / 68.3 us (k_mg_pre0_w 6.6 / 4.7, k_mg_post0_w 8.5 / 5.8), 652,000 unknowns 99.1 / 95.7,
// 842,000 109.6 / 107.7, 1,287,000 122.0 / 126.7, 1,645,000 125.1 / 131.0 us.
constexpr int kMgSplitBricks = 2048;

#define SHK_MG_LAUNCH0(kernel, op, ...)                                                            \
    do {                                                                                           \
        const bool split = (op).n_active <= kMgSplitBricks;                                        \
        const dim3 grid(blocks((int64_t)(op).n_active * (split ? 256 : 64))), block(NT);           \
        if ((op).bx == 64 && split)                                                                \
            hipLaunchKernelGGL((kernel<64, 2>), grid, block, 0, __VA_ARGS__);                      \
        else if ((op).bx == 64)                                                                    \
            hipLaunchKernelGGL((kernel<64, 8>), grid, block, 0, __VA_ARGS__);                      \
        else if (split)                                                                            \
            hipLaunchKernelGGL((kernel<8, 2>), grid, block, 0, __VA_ARGS__);                       \
        else                                                                                       \
            hipLaunchKernelGGL((kernel<8, 8>), grid, block, 0, __VA_ARGS__);                       \
    } while (0)

void launch_mg_pre0(hipStream_t st, const MgOp &op, const float *r, const int4 *coord, const int *parent,
                    const MgLevelDev &c1, float omega_c, const SolveState *state) {
    SHK_MG_LAUNCH0(k_mg_pre0_w, op, st, op, r, coord, parent, c1, omega_c, state);
}

int mg_partials(int n_active) {
    const int nb = (int)blocks((int64_t)n_active * (n_active <= kMgSplitBricks ? 256 : 64));
    return nb <= kMgMaxPartials ? nb : kMaxBlocks;
}

void launch_mg_post0(hipStream_t st, const MgOp &op, const int4 *coord, const int *parent, const float *r,
                     const float *xc, float *y, const SolveState *state, double *cell_part, double *part) {
    const int nb = (int)blocks((int64_t)op.n_active * (op.n_active <= kMgSplitBricks ? 256 : 64));
    const bool fold = nb > kMgMaxPartials;
    SHK_MG_LAUNCH0(k_mg_post0_w, op, st, op, coord, parent, r, xc, y, state, fold ? cell_part : part);
    if (fold)
        hipLaunchKernelGGL(k_mg_fold, dim3((kMaxBlocks + NT - 1) / NT), dim3(NT), 0, st, nb, cell_part, kMaxBlocks,
                           part, state);
}

void launch_mg_tail(hipStream_t st, int bx, const MgTail &t, float omega, float alpha, const SolveState *state) {
    if (bx == 64)
        hipLaunchKernelGGL(k_mg_tail<64>, dim3(1), dim3(TNT), 0, st, t, omega, alpha, state);
    else
        hipLaunchKernelGGL(k_mg_tail<8>, dim3(1), dim3(TNT), 0, st, t, omega, alpha, state);
}

}  // namespace shk
