// resident.hip -- the whole CG solve of a brick system in one launch (see krylov.h).
//
// What bounds the two-kernel iteration (krylov.hip) depends on the size.  Small systems:
// two launches of about 5 us each however little they do (fold of the partials, loads,
// stores, one after another).  Systems that fit the caches: ten vector streams per
// iteration, 52 bytes per cell in FP32.  One MI355X holds 128 MB of vector registers and
// 40 MB of LDS, so up to a few million unknowns the four CG vectors fit on the chip:
// here every wave keeps its bricks' r, s and q in registers (x too when they leave room,
// else in LDS) for the whole solve, and one iteration moves only the brick faces:
//   sigma = s.q            grid-wide exchange 1 (also: nobody reads old faces any more)
//   x += alpha s; r -= alpha q; the faces of r go to memory
//   rho = r.r, max|r|      grid-wide exchange 2 (also: the faces of r have arrived)
//   the neighbours' faces of r are read; s = r + beta s, and the same on the halo planes
//   of s, which stay in registers; q = A s
// The arithmetic per cell is k_dir_spmv's and k_axpy_norm's; only the order in which the
// partial sums are folded differs (one fixed order per launch shape, the same in every
// workgroup).
//
// Exchange: each workgroup publishes its pair of partials in its own slot and one wave of
// every workgroup polls all slots (a slot that holds the sentinel has not arrived yet),
// so one exchange costs one store and one load through memory instead of a counter and
// a second read.  Four slot sets rotate: passing exchange e proves that everybody has
// finished reading set e - 2 = e + 2 (mod 4), which is cleared then.  Slots and faces are
// written and read with agent-scope accesses (past the XCDs' private L2s); a workgroup's
// face stores are complete (vmcnt 0 in every wave) before it arrives.
//
// Measured against the two-kernel iteration, whole projections to 1e-6: 32x36x28 mixed
// Jacobi 2.38 -> 0.90 ms, 100x77x90 FP64 Jacobi 6.9 -> 2.8 ms, 256^3 mixed Jacobi 32.1 ->
// 13.3 ms, 600x450 (2D) mixed Jacobi 20.3 -> 7.2 ms.  One iteration at 256^3 takes 48.5
// thousand cycles (52 us before): 14.6 the stencil (11 to 18 by the bricks a workgroup has),
// 18.6 the two exchanges with the wait for the slowest workgroup, 6.8 the halo planes, 8.6 the
// update and the faces.
//
// All workgroups have to be on the chip at once.  A launch takes at most one workgroup
// per CU and the launches of a process share that budget (CuBudget), but another process
// or a CU mask can keep a part of the workgroups out.  So a wait that lasts its limit
// gives up: every workgroup then leaves, the state says aborted, the caller runs the
// two-kernel solve, and the context leaves this form alone for a number of solves that
// doubles with every further give-up (OneLaunchRest): 0.67 s of waiting for each 10 ms
// solve would be paid on every call otherwise.
#include <hip/hip_runtime.h>

#include "cu_budget.h"
#include "krylov.h"
#include "shk_projection.h"

namespace shk {

namespace {

constexpr int RT = 512;               // threads of a workgroup: 8 waves, 2 per SIMD
constexpr int RW = RT / kWave;        // waves of a workgroup
constexpr int NT = kBrickCells;
constexpr int kMaxWg = 256;           // slots of one exchange
// Every slot has kRep copies, and workgroup g polls copy g % kRep: with one copy 256 polling
// workgroups wait for the same few cache lines (2.8 us per exchange; 2.0 with 4 to 16
// copies; 32 workgroups 1.9 and 1.45).  The copies' spacing keeps them off one memory
// channel.  A slot is a pair of words, kMaxWg apart: sum and maximum.
constexpr int kRep = 8;
constexpr int kRepWords = 2 * kMaxWg + 32, kSetWords = kRep * kRepWords, kSlotWords = 4 * kSetWords;
constexpr int kCsrW = 8;              // entries of a CSR row held in registers
constexpr unsigned long long kEmpty = 0xFFF8DEADBEEF0001ull;  // a NaN that no sum produces
constexpr double kTicksPerSecond = 1e8;  // s_memrealtime; 32 bits of it are 42 s

__device__ inline void st_agent(unsigned long long *p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long ld_agent(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_face(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_face(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ inline T ld_face(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int CTRL>
__device__ inline double dpp64(double v) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true));
}
__device__ inline double lane_of(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// Sum / maximum over the wave, the same in every lane: DPP moves within the rows of 16
// (neighbours, pairs, half rows, rows), then the four rows in order.  The shuffles of
// wave_sum take about five times as long, and an exchange has two of these in a row.
struct OpAdd {
    __device__ static double f(double a, double b) { return a + b; }
};
struct OpMax {
    __device__ static double f(double a, double b) { return fmax(a, b); }
};
template <class OP>
__device__ inline double wave_all(double v) {
    v = OP::f(v, dpp64<0xB1>(v));   // quad_perm 1,0,3,2
    v = OP::f(v, dpp64<0x4E>(v));   // quad_perm 2,3,0,1
    v = OP::f(v, dpp64<0x141>(v));  // row_half_mirror
    v = OP::f(v, dpp64<0x140>(v));  // row_mirror
    return OP::f(OP::f(lane_of(v, 0), lane_of(v, 16)), OP::f(lane_of(v, 32), lane_of(v, 48)));
}

struct ExchLds {
    double sum[RW], mx[RW];
    double tot[2];
    int gone;
    uint32_t limit;  // clock ticks until a wait gives up (here, not in a register kept for it)
};

// Sum of `v` (and, with MAX, the maximum of `m`) over the grid, the same bits in every
// thread; false when a wait gave up.  Every memory access issued before is complete when
// others pass.
template <bool MAX>
__device__ inline bool exchange(double v, double m, unsigned e, unsigned long long *slots, ExchLds &l, double &sum,
                                double &mx) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, G = gridDim.x;
    v = wave_all<OpAdd>(v);
    if constexpr (MAX) m = wave_all<OpMax>(m);
    if (lane == 0) {
        l.sum[wave] = v;
        if constexpr (MAX) l.mx[wave] = m;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (wave == 0) {
        double ps = 0.0, pm = 0.0;
#pragma unroll
        for (int w = 0; w < RW; ++w) {
            ps += l.sum[w];
            if constexpr (MAX) pm = fmax(pm, l.mx[w]);
        }
        int gone = 0;
        if (G > 1) {
            // lanes 0..7 store the sum's copies, lanes 8..15 the maximum's
            const int copy = (lane & (kRep - 1)) * kRepWords + (lane >= kRep ? kMaxWg : 0) + blockIdx.x;
            unsigned long long *set = slots + (size_t)(e & 3) * kSetWords;
            if (lane < (MAX ? 2 : 1) * kRep) {
                unsigned long long bits = (unsigned long long)__double_as_longlong(lane >= kRep ? pm : ps);
                if (bits == kEmpty) bits ^= 2;
                st_agent(set + copy, bits);
            }
            const unsigned long long *mine = set + (size_t)(blockIdx.x % kRep) * kRepWords;
            unsigned long long a[kMaxWg / kWave], b[kMaxWg / kWave];
            const unsigned long long end =
                __builtin_amdgcn_s_memrealtime() + (uint32_t)__builtin_amdgcn_readfirstlane((int)l.limit);
            for (;;) {
                bool ok = true;
#pragma unroll
                for (int c = 0; c < kMaxWg / kWave; ++c) {
                    a[c] = b[c] = 0ull;
                    const int w = lane + kWave * c;
                    if (w < G) {
                        a[c] = ld_agent(mine + w);
                        if constexpr (MAX) b[c] = ld_agent(mine + kMaxWg + w);
                    }
                }
#pragma unroll
                for (int c = 0; c < kMaxWg / kWave; ++c) ok = ok && a[c] != kEmpty && b[c] != kEmpty;
                if (__all(ok)) break;
                if (__builtin_amdgcn_s_memrealtime() > end) {
                    gone = 1;
                    break;
                }
            }
            // this workgroup's slot of the set that exchange e + 2 uses
            if (lane < 2 * kRep) st_agent(slots + (size_t)((e + 2) & 3) * kSetWords + copy, kEmpty);
            ps = pm = 0.0;
#pragma unroll
            for (int c = 0; c < kMaxWg / kWave; ++c) {
                ps += __longlong_as_double((long long)a[c]);
                if constexpr (MAX) pm = fmax(pm, __longlong_as_double((long long)b[c]));
            }
            ps = wave_all<OpAdd>(ps);
            if constexpr (MAX) pm = wave_all<OpMax>(pm);
        }
        if (lane == 0) {
            l.tot[0] = ps;
            l.tot[1] = pm;
            l.gone = gone;
        }
    }
    __syncthreads();
    sum = l.tot[0];
    if constexpr (MAX) mx = l.tot[1];
    return l.gone == 0;
}

template <class T>
__device__ inline T lane_get(T v, int src) {
    return __shfl(v, src & (kWave - 1), kWave);
}

// the value of the lane before (CTRL 0x138, wave_shr:1) or after (0x130, wave_shl:1): a DPP
// move, no LDS access; the ends get 0 (a halo value replaces them)
template <int CTRL>
__device__ inline float lane_shift(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ inline double lane_shift(double v) {
    return dpp64<CTRL>(v);
}

// Hides a wave-uniform value's origin, so that the addresses formed from it are computed
// where they are used (scalar instructions) and not kept in registers through the solve.
__device__ inline int here(int v) {
    asm volatile("" : "+s"(v));
    return v;
}

// acc += v, with PIN not moved behind later cells: the compiler would otherwise keep every
// cell's factors as doubles (two registers each) until the end of the brick
template <bool PIN>
__device__ inline void add_here(double &acc, double v) {
    acc += v;
    if constexpr (PIN) asm volatile("" : "+v"(acc));
}

// LDS accesses of one wave are executed in order: keep the compiler from moving them
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The brick's face planes of r for the neighbours that exist: x planes as (y = a, z = c) at
// a + Y c, y planes as (x = a, z = c) at a + X c, z planes (x, y) at the lane.  The lateral
// planes lie across registers and lanes: they pass through the wave's LDS scratch.
template <class T, int BX>
__device__ inline void publish(const T (&r)[8], T *scr, T *face, int lane, const int (&nb)[6]) {
    using B = BrickShape<BX>;
    constexpr int X = B::X, Y = B::Y;
    const int i = lane % X, j = lane / X;
    if (i == 0 || i == X - 1) {
        T *p = scr + (i ? 64 : 0) + j;
#pragma unroll
        for (int k = 0; k < 8; ++k) p[Y * k] = r[k];
    }
    if constexpr (Y > 1) {
        if (j == 0 || j == Y - 1) {
            T *p = scr + (j ? 192 : 128) + i;
#pragma unroll
            for (int k = 0; k < 8; ++k) p[X * k] = r[k];
        }
    }
    wave_lds_fence();
    const bool xl = lane < Y * 8;
    if (nb[0] >= 0 && xl) st_face(face + lane, scr[lane]);
    if (nb[1] >= 0 && xl) st_face(face + 64 + lane, scr[64 + lane]);
    if constexpr (Y > 1) {
        if (nb[2] >= 0) st_face(face + 128 + lane, scr[128 + lane]);
        if (nb[3] >= 0) st_face(face + 192 + lane, scr[192 + lane]);
    }
    if (nb[4] >= 0) st_face(face + 256 + lane, r[0]);
    if (nb[5] >= 0) st_face(face + 320 + lane, r[7]);
    wave_lds_fence();
}

// The couplings of a cell column: low x, high x, low y, high y, low z (the high z ones are
// the next cell's low ones; c.top is the one above the brick) and the diagonal.
template <class T, bool UNIT>
struct Couplings {
    T x[8], xp[8], y[8], yp[8], z[8], top, d[UNIT ? 1 : 8];
};
// where they lie, as 32-bit byte offsets (a resident system is far below 4 GB); a cell's +x /
// +y coupling is its neighbour's low one, in the next brick for the edge lanes (without one
// the halo value is 0, and any finite coupling will do)
template <class T, bool UNIT, int BX>
struct CouplingAt {
    const char *cx, *cy, *cz, *dg;
    uint32_t own, xp, yp, up;
    bool open;
    __device__ CouplingAt(const BrickOp<T> &op, int slot, const int (&nb)[6], int lane) {
        constexpr int X = BrickShape<BX>::X, Y = BrickShape<BX>::Y;
        const int i = lane % X, j = lane / X;
        cx = (const char *)op.cx;
        cy = (const char *)op.cy;
        cz = (const char *)op.cz;
        dg = (const char *)op.diag;
        const int base = slot * NT;
        open = nb[5] >= 0;
        const int xi = i < X - 1 ? base + lane + 1 : (nb[1] >= 0 ? nb[1] * NT + X * j : base + lane);
        const int yi = j < Y - 1 ? base + lane + X : (nb[3] >= 0 ? nb[3] * NT + i : base + lane);
        own = (uint32_t)(base + lane) * (uint32_t)sizeof(T);
        xp = (uint32_t)xi * (uint32_t)sizeof(T);
        yp = (uint32_t)yi * (uint32_t)sizeof(T);
        up = (uint32_t)((open ? nb[5] : slot) * NT + lane) * (uint32_t)sizeof(T);
    }
    __device__ static T at(const char *p, uint32_t off, int k) {
        return *reinterpret_cast<const T *>(p + off + 64 * k * (int)sizeof(T));
    }
    __device__ void load(Couplings<T, UNIT> &c, int k) const {
        constexpr int Y = BrickShape<BX>::Y;
        c.x[k] = at(cx, own, k);
        c.xp[k] = at(cx, xp, k);
        c.y[k] = Y > 1 ? at(cy, own, k) : T(0);
        c.yp[k] = Y > 1 ? at(cy, yp, k) : T(0);
        c.z[k] = at(cz, own, k);
        if (!UNIT) c.d[UNIT ? 0 : k] = at(dg, own, k);
        if (k == 7) c.top = open ? at(cz, up, 0) : T(0);
    }
};

// Whether a solve ends before its first iteration: zero rhs, rho == 0, NaN (pcg_solver.h:
// 254-271, as k_finish_init)
__device__ inline bool start_state(double rho, double rnorm0, int64_t max_iter, int &status) {
    if (rnorm0 == 0.0) return true;
    if (rho == 0.0) {
        status = SHK_BREAKDOWN;
    } else if (rho != rho) {
        status = SHK_NAN;
    } else if (max_iter <= 0) {
        status = SHK_NOT_CONVERGED;
    } else {
        return false;
    }
    return true;
}
// The stop test of pcg_solver.h:281-284 and beta of :287-289 (as direction_step): true when
// the solve has stopped
__device__ inline bool next_direction(double rho_new, double rn, double tol_abs, int64_t it, int64_t max_iter,
                                      double &rho, double &beta, int &status) {
    if (rn <= tol_abs) return true;
    if (rho_new != rho_new) {
        status = SHK_NAN;
    } else if (it >= max_iter) {
        status = SHK_NOT_CONVERGED;
    } else {
        beta = rho_new / rho;
        rho = rho_new;
        return false;
    }
    return true;
}
__device__ inline void end_state(SolveState *st, bool alive, double rho, double alpha, double beta, double sigma,
                                 double rn, double rnorm0, double tol_abs, int64_t it, int64_t max_iter, int status) {
    // a wait that gave up is seen by some workgroups only: any of them says so, and the rest
    // of the state counts for nothing
    if (threadIdx.x != 0) return;
    if (blockIdx.x == 0) {
        st->rho_k1 = rho;
        st->rho_k2 = rho;
        st->alpha = alpha;
        st->beta = beta;
        st->sigma = sigma;
        st->rnorm = rn;
        st->rnorm0 = rnorm0;
        st->tol_abs = tol_abs;
        st->iter = it;
        st->max_iter = max_iter;
        st->done = 1;
        st->status = status;
    }
    if (!alive) st->aborted = 1;
}

template <class T, bool UNIT, int BX, bool SCALED, int BPW>
__global__ __launch_bounds__(RT, 2) void k_cg_resident(BrickOp<T> op, const T *__restrict__ rhs,
                                                       const double *__restrict__ sig, T *__restrict__ xout,
                                                       T *__restrict__ faces, unsigned long long *__restrict__ slots,
                                                       SolveState *__restrict__ st, double tol_rel, int64_t max_iter,
                                                       uint32_t limit) {
    using B = BrickShape<BX>;
    constexpr int X = B::X, Y = B::Y;
    // with few bricks x and the couplings stay in registers too; else the couplings are read
    // every iteration (they stay in the L2s), two cells of a column ahead of their use
    constexpr bool XREG = BPW * (int)sizeof(T) <= 8, CREG = XREG;
    constexpr int NC = CREG ? BPW : 1;
    __shared__ ExchLds xl_;
    __shared__ T scratch[RW][256];
    __shared__ T halo[RW * BPW][256];  // the lateral halo planes of s (-x, +x, -y, +y)
    __shared__ T xs[XREG ? 1 : RW * BPW * NT];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = lane % X, j = lane / X;
    const bool xl = lane < Y * 8;
    // bricks blockIdx + G (wave + 8 b): those with couplings of their own lie together (walls,
    // the surface) and cost several times a uniform brick, so they are dealt out one by one
    const int slot0 = blockIdx.x + gridDim.x * wave, stride = gridDim.x * RW;
    T *scr = scratch[wave];
    // where an edge lane reads its halo value of z = k: + Y k (x planes), + X k (y planes)
    const int hxo = (i == 0 ? 0 : 64) + j, hyo = (j == 0 ? 128 : 192) + i;
    const bool xlo = i == 0, xhi = i == X - 1, ylo = j == 0, yhi = j == Y - 1;
    T r[BPW][8], s[BPW][8], q[BPW][8], hz[BPW][2], x[XREG ? BPW : 1][8];
    int nb[BPW][6];
    T kap[BPW], kd[BPW];
    Couplings<T, UNIT> cpl[NC];
    T isg[SCALED && CREG ? BPW : 1][8];  // 1 / sig for the stop test
    unsigned e = 0;
    double acc = 0.0, mx = 0.0;
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
        const int slot = slot0 + stride * b;
        const bool on = slot < op.n_active;
#pragma unroll
        for (int f = 0; f < 6; ++f) nb[b][f] = on ? __builtin_amdgcn_readfirstlane(op.nbr[6 * slot + f]) : -1;
        hz[b][0] = hz[b][1] = T(0);
        kap[b] = on ? op.kappa[slot] : T(1);
        kd[b] = !UNIT && on ? op.kdiag[slot] : T(0);
        if constexpr (CREG)
            if (kap[b] == T(0)) {
                const CouplingAt<T, UNIT, BX> at(op, slot, nb[b], lane);
#pragma unroll
                for (int k = 0; k < 8; ++k) at.load(cpl[CREG ? b : 0], k);
            }
#pragma unroll
        for (int f = 0; f < 4; ++f) halo[wave * BPW + b][64 * f + lane] = T(0);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            T rv = T(0);
            if (on) {
                const T bv = (rhs + (int64_t)slot * NT)[lane + 64 * k];
                const double sg = SCALED ? (sig + (int64_t)slot * NT)[lane + 64 * k] : 1.0;
                rv = SCALED ? (T)(sg * (double)bv) : bv;
                if constexpr (SCALED && CREG) isg[b][k] = sg > 0.0 ? (T)(1.0 / sg) : T(0);
                // with a scaled system the stop test is on the unscaled residual: max|b|
                mx = fmax(mx, SCALED ? (sg > 0.0 ? fabs((double)bv) : 0.0) : fabs((double)rv));
            }
            r[b][k] = s[b][k] = rv;
            q[b][k] = T(0);
            if constexpr (XREG)
                x[b][k] = T(0);
            else
                xs[((wave * BPW + b) * 8 + k) * 64 + lane] = T(0);
            acc += (double)rv * (double)rv;
        }
        if (on) publish<T, BX>(r[b], scr, faces + (int64_t)slot * 384, lane, nb[b]);
    }
    double rho = 0.0, rn = 0.0, sigma = 0.0, alpha = 0.0, beta = 0.0;
    if (threadIdx.x == 0) xl_.limit = limit;
    bool alive = exchange<true>(acc, mx, e++, slots, xl_, rho, rn) && limit != 0;  // 0: all give up
    const double rnorm0 = rn;
    const double tol_abs = (tol_rel < 1e-30 ? 1e-30 : tol_rel) * rnorm0;  // pcg_solver.h:235
    int64_t it = 0;
    int status = SHK_OK;
    bool done = start_state(rho, rnorm0, max_iter, status) || !alive;
    while (!done) {
        // the neighbours' faces of r: s = r + beta s on the halo planes and the cells
        const T bt = (T)beta;
        if constexpr (!CREG)
            if (kap[0] == T(0)) {
                int n[6];
#pragma unroll
                for (int f = 0; f < 6; ++f) n[f] = here(nb[0][f]);
                const CouplingAt<T, UNIT, BX> at(op, here(slot0), n, lane);
                at.load(cpl[0], 0);
                at.load(cpl[0], 1);
            }
        constexpr int HG = BPW > 4 ? (BPW + 1) / 2 : BPW;  // bricks whose faces are in flight at once
        if (it > 0) {  // the first direction is r itself
#pragma unroll
            for (int b = 0; b < BPW; ++b)
#pragma unroll
                for (int k = 0; k < 8; ++k) s[b][k] = r[b][k] + bt * s[b][k];
        }
#pragma unroll
        for (int g = 0; g < BPW; g += HG) {
            __builtin_amdgcn_sched_barrier(0);
            T hr[HG][6];
#pragma unroll
            for (int u = 0; u < HG; ++u) {
                const int b = g + u < BPW ? g + u : g;
                int n[6];
#pragma unroll
                for (int f = 0; f < 6; ++f) n[f] = here(nb[b][f]);
                hr[u][0] = n[0] >= 0 && xl ? ld_face(faces + (int64_t)n[0] * 384 + 64 + lane) : T(0);
                hr[u][1] = n[1] >= 0 && xl ? ld_face(faces + (int64_t)n[1] * 384 + lane) : T(0);
                hr[u][2] = hr[u][3] = T(0);
                if constexpr (Y > 1) {
                    hr[u][2] = n[2] >= 0 ? ld_face(faces + (int64_t)n[2] * 384 + 192 + lane) : T(0);
                    hr[u][3] = n[3] >= 0 ? ld_face(faces + (int64_t)n[3] * 384 + 128 + lane) : T(0);
                }
                hr[u][4] = n[4] >= 0 ? ld_face(faces + (int64_t)n[4] * 384 + 320 + lane) : T(0);
                hr[u][5] = n[5] >= 0 ? ld_face(faces + (int64_t)n[5] * 384 + 256 + lane) : T(0);
            }
#pragma unroll
            for (int u = 0; u < HG; ++u) {
                if (g + u >= BPW) continue;
                const int b = g + u < BPW ? g + u : g;
                T *hp = halo[wave * BPW + b];
#pragma unroll
                for (int f = 0; f < (Y > 1 ? 4 : 2); ++f) hp[64 * f + lane] = hr[u][f] + bt * hp[64 * f + lane];
                hz[b][0] = hr[u][4] + bt * hz[b][0];
                hz[b][1] = hr[u][5] + bt * hz[b][1];
            }
        }
        wave_lds_fence();
        acc = 0.0;
#pragma unroll
        for (int b = 0; b < BPW; ++b) {
            __builtin_amdgcn_sched_barrier(0);  // one brick at a time: registers
            const int slot = here(slot0) + stride * b;
            if (slot >= op.n_active) continue;
            const T *hp = halo[wave * BPW + b];
            const bool next = !CREG && b + 1 < BPW && slot + stride < op.n_active && kap[b + 1 < BPW ? b + 1 : b] == T(0);
            int nn[6];
            if constexpr (!CREG) {
#pragma unroll
                for (int f = 0; f < 6; ++f) nn[f] = here(nb[b + 1 < BPW ? b + 1 : b][f]);
            }
            if (kap[b] != T(0)) {
                if (next) {
                    const CouplingAt<T, UNIT, BX> at(op, slot + stride, nn, lane);
                    at.load(cpl[0], 0);
                    at.load(cpl[0], 1);
                }
                const T kv = kap[b];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    if constexpr (!CREG)
                        if ((k & 1) == 0) __builtin_amdgcn_sched_barrier(0);
                    const T sk = s[b][k];
                    const T hx = hp[hxo + Y * k];
                    const T lf = lane_shift<0x138>(sk), rt = lane_shift<0x130>(sk);  // every lane takes part
                    const T xm = xlo ? hx : lf, xp = xhi ? hx : rt;
                    T ym = T(0), yp = T(0);
                    if constexpr (Y > 1) {
                        const T hy = hp[hyo + X * k];
                        const T dn = lane_get(sk, lane - X), up = lane_get(sk, lane + X);
                        ym = ylo ? hy : dn;
                        yp = yhi ? hy : up;
                    }
                    const T zm = k > 0 ? s[b][k - 1] : hz[b][0];
                    const T zp = k < 7 ? s[b][k + 1] : hz[b][1];
                    T qv = UNIT ? sk : kd[b] * sk;
                    qv -= kv * xm + kv * xp + kv * ym + kv * yp + kv * zm + kv * zp;
                    q[b][k] = qv;
                    add_here<!CREG>(acc, (double)sk * (double)qv);
                }
                continue;
            }
            Couplings<T, UNIT> &c = cpl[CREG ? b : 0];
            int n[6];
#pragma unroll
            for (int f = 0; f < 6; ++f) n[f] = CREG ? -1 : here(nb[b][f]);
            const CouplingAt<T, UNIT, BX> at(op, slot, n, lane);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if constexpr (!CREG)
                    if ((k & 1) == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (k < 6) {
                            at.load(c, k + 2 < 8 ? k + 2 : 7);
                            at.load(c, k + 3 < 8 ? k + 3 : 7);
                        }
                    }
                const T sk = s[b][k];
                const T hx = hp[hxo + Y * k];
                const T lf = lane_shift<0x138>(sk), rt = lane_shift<0x130>(sk);
                const T xm = xlo ? hx : lf, xp = xhi ? hx : rt;
                T ym = T(0), yp = T(0);
                if constexpr (Y > 1) {
                    const T hy = hp[hyo + X * k];
                    const T dn = lane_get(sk, lane - X), up = lane_get(sk, lane + X);
                    ym = ylo ? hy : dn;
                    yp = yhi ? hy : up;
                }
                const T zm = k > 0 ? s[b][k - 1] : hz[b][0];
                const T zp = k < 7 ? s[b][k + 1] : hz[b][1];
                const T czp = k < 7 ? c.z[k < 7 ? k + 1 : 7] : c.top;
                T qv = UNIT ? sk : c.d[UNIT ? 0 : k] * sk;
                qv -= c.x[k] * xm + c.xp[k] * xp + c.y[k] * ym + c.yp[k] * yp + c.z[k] * zm + czp * zp;
                q[b][k] = qv;
                add_here<!CREG>(acc, (double)sk * (double)qv);
                if constexpr (!CREG)
                    if (k == 5 && next) {
                        const CouplingAt<T, UNIT, BX> an(op, slot + stride, nn, lane);
                        an.load(cpl[0], 0);
                        an.load(cpl[0], 1);
                    }
            }
        }
        if (!(alive = exchange<false>(acc, 0.0, e++, slots, xl_, sigma, mx))) break;
        if (!(sigma > 0.0)) {
            status = sigma != sigma ? SHK_NAN : SHK_BREAKDOWN;
            break;
        }
        alpha = rho / sigma;
        ++it;
        const T a = (T)alpha;
        acc = 0.0;
        mx = 0.0;
#pragma unroll
        for (int b = 0; b < BPW; ++b) {
            __builtin_amdgcn_sched_barrier(0);
            const int slot = here(slot0) + stride * b;
            if (slot >= op.n_active) continue;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if constexpr (XREG)
                    x[b][k] += a * s[b][k];
                else
                    xs[((wave * BPW + b) * 8 + k) * 64 + lane] += a * s[b][k];
                const T rv = r[b][k] - a * q[b][k];
                r[b][k] = rv;
                add_here<!CREG>(acc, (double)rv * (double)rv);
                if constexpr (SCALED) {
                    T is;
                    if constexpr (CREG) {
                        is = isg[b][k];
                    } else {
                        const double sg = (sig + (int64_t)slot * NT)[lane + 64 * k];
                        is = sg > 0.0 ? (T)(1.0 / sg) : T(0);
                    }
                    mx = fmax(mx, fabs((double)(rv * is)));
                } else {
                    mx = fmax(mx, fabs((double)rv));
                }
            }
            int n[6];
#pragma unroll
            for (int f = 0; f < 6; ++f) n[f] = here(nb[b][f]);
            publish<T, BX>(r[b], scr, faces + (int64_t)slot * 384, lane, n);
        }
        double rho_new;
        if (!(alive = exchange<true>(acc, mx, e++, slots, xl_, rho_new, rn))) break;
        done = next_direction(rho_new, rn, tol_abs, it, max_iter, rho, beta, status);
    }
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
        const int slot = slot0 + stride * b;
        if (slot >= op.n_active) continue;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            (xout + (int64_t)slot * NT)[lane + 64 * k] = XREG ? x[XREG ? b : 0][k]
                                                            : xs[XREG ? 0 : ((wave * BPW + b) * 8 + k) * 64 + lane];
    }
    end_state(st, alive, rho, alpha, beta, sigma, rn, rnorm0, tol_abs, it, max_iter, status);
}

// ---------------------------------------------------------------- CSR

// The same solve for a CSR matrix of rows with at most kCsrW entries: a thread keeps RPT rows,
// their entries (32-bit columns) and, instead of halo planes, the value of s at each entry's
// column, which it updates from the gathered r exactly as the column's own thread does.  An
// iteration then moves one publication and one gather of r and no matrix: the two-kernel
// iteration read 16 bytes per entry and gathered r and s.  288,000 rows of 7, solve: 12.0 ms
// with two kernels an iteration (26 us), 3.57 ms here (7.6 us: two exchanges and the gather).
// The system is the Jacobi-scaled D^-1/2 A D^-1/2 (values as k_csr_scale forms them), the
// stop test is on the unscaled residual, and x is scaled back at the end.
template <int RPT>
__global__ __launch_bounds__(RT, 2) void k_csr_resident(CsrOp op, const double *__restrict__ rhs,
                                                        const double *__restrict__ sig, double *__restrict__ xout,
                                                        double *__restrict__ pub, unsigned long long *__restrict__ slots,
                                                        SolveState *__restrict__ st, double tol_rel, int64_t max_iter,
                                                        uint32_t limit) {
    constexpr int W = kCsrW;
    __shared__ ExchLds xl_;
    const int row0 = blockIdx.x * (RT * RPT) + threadIdx.x, rows = (int)op.rows;
    double val[RPT][W], sn[RPT][W], x[RPT], r[RPT], s[RPT], q[RPT], isg[RPT];
    int col[RPT][W];
    unsigned e = 0;
    double acc = 0.0, mx = 0.0;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int row = row0 + RT * k;
        const bool on = row < rows;
        const double sg = on ? sig[row] : 0.0, b = on ? rhs[row] : 0.0;
        const int64_t p0 = on ? op.rowptr[row] : 0, p1 = on ? op.rowptr[row + 1] : 0;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const bool in = p0 + j < p1;
            col[k][j] = in ? (int)op.cols[p0 + j] : (on ? row : 0);
            val[k][j] = in ? sg * op.vals[p0 + j] * sig[col[k][j]] : 0.0;
            sn[k][j] = 0.0;
        }
        isg[k] = sg > 0.0 ? 1.0 / sg : 0.0;
        x[k] = 0.0;
        r[k] = s[k] = sg * b;
        q[k] = 0.0;
        acc += r[k] * r[k];
        mx = fmax(mx, sg > 0.0 ? fabs(b) : 0.0);
        if (on) st_face(pub + row, r[k]);
    }
    double rho = 0.0, rn = 0.0, sigma = 0.0, alpha = 0.0, beta = 0.0;
    if (threadIdx.x == 0) xl_.limit = limit;
    bool alive = exchange<true>(acc, mx, e++, slots, xl_, rho, rn) && limit != 0;  // 0: all give up
    const double rnorm0 = rn;
    const double tol_abs = (tol_rel < 1e-30 ? 1e-30 : tol_rel) * rnorm0;  // pcg_solver.h:235
    int64_t it = 0;
    int status = SHK_OK;
    bool done = start_state(rho, rnorm0, max_iter, status) || !alive;
    while (!done) {
        double g[RPT][W];
#pragma unroll
        for (int k = 0; k < RPT; ++k)
#pragma unroll
            for (int j = 0; j < W; ++j) g[k][j] = ld_face(pub + col[k][j]);
        acc = 0.0;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            if (it > 0) s[k] = r[k] + beta * s[k];
            double a = 0.0;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                sn[k][j] = g[k][j] + beta * sn[k][j];
                a += val[k][j] * sn[k][j];
            }
            q[k] = a;
            acc += s[k] * a;
        }
        if (!(alive = exchange<false>(acc, 0.0, e++, slots, xl_, sigma, mx))) break;
        if (!(sigma > 0.0)) {
            status = sigma != sigma ? SHK_NAN : SHK_BREAKDOWN;
            break;
        }
        alpha = rho / sigma;
        ++it;
        acc = 0.0;
        mx = 0.0;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            x[k] += alpha * s[k];
            r[k] = r[k] - alpha * q[k];
            acc += r[k] * r[k];
            mx = fmax(mx, fabs(r[k] * isg[k]));
            if (row0 + RT * k < rows) st_face(pub + row0 + RT * k, r[k]);
        }
        double rho_new;
        if (!(alive = exchange<true>(acc, mx, e++, slots, xl_, rho_new, rn))) break;
        done = next_direction(rho_new, rn, tol_abs, it, max_iter, rho, beta, status);
    }
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int row = row0 + RT * k;
        if (row < rows) xout[row] = x[k] * sig[row];
    }
    end_state(st, alive, rho, alpha, beta, sigma, rn, rnorm0, tol_abs, it, max_iter, status);
}

__global__ void k_resident_begin(SolveState *st, unsigned long long *slots) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kSlotWords) slots[i] = kEmpty;
    if (i == 0) st->aborted = 0;
}

constexpr int kMaxDevices = 64;
CuBudget g_budget[kMaxDevices];

// Bricks per wave the kernels are built for.  The registers of a wave at 2 waves per SIMD
// (256) hold 6 FP32 bricks (r, s, q and the halo of s: 30 each) or 2 FP64 ones.
constexpr int kBpwF32[] = {1, 2, 3, 4, 6};
constexpr int kBpwF64[] = {1, 2};

template <class T, bool UNIT, int BX, bool SCALED, int BPW>
void launch_one(hipStream_t st, int blocks, const BrickOp<T> &op, const T *rhs, const double *sig, T *x, T *faces,
                unsigned long long *slots, SolveState *state, double tol_rel, int64_t max_iter, uint32_t limit) {
    hipLaunchKernelGGL((k_cg_resident<T, UNIT, BX, SCALED, BPW>), dim3(blocks), dim3(RT), 0, st, op, rhs, sig, x,
                       faces, slots, state, tol_rel, max_iter, limit);
}

template <class T, bool UNIT, int BX, bool SCALED>
void launch_bpw(hipStream_t st, const ResidentPlan &p, const BrickOp<T> &op, const T *rhs, const double *sig, T *x,
                T *faces, unsigned long long *slots, SolveState *state, double tol_rel, int64_t max_iter,
                uint32_t limit) {
#define SHK_RES(N)                                                                                                  \
    case N:                                                                                                         \
        launch_one<T, UNIT, BX, SCALED, N>(st, p.blocks, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter,   \
                                           limit);                                                                 \
        break
    if constexpr (sizeof(T) == 4) {
        switch (p.bpw) {
            SHK_RES(1);
            SHK_RES(2);
            SHK_RES(3);
            SHK_RES(4);
            SHK_RES(6);
        }
    } else {
        switch (p.bpw) {
            SHK_RES(1);
            SHK_RES(2);
        }
    }
#undef SHK_RES
}

}  // namespace

size_t resident_slot_words() { return kSlotWords; }

template <class T>
ResidentPlan resident_plan(const BrickOp<T> &op, int device, int cus) {
    ResidentPlan p;
    if (device < 0 || device >= kMaxDevices || op.n_active < 1 || !op.kappa || (op.diag && !op.kdiag)) return p;
    const int cap = cus < kMaxWg ? cus : kMaxWg;
    auto fits = [&](int bpw) {
        const int blocks = (op.n_active + RW * bpw - 1) / (RW * bpw);
        if (blocks > cap) return false;
        p.bpw = bpw;
        p.blocks = blocks;
        return true;
    };
    if constexpr (sizeof(T) == 4) {
        for (int b : kBpwF32)
            if (fits(b)) break;
    } else {
        for (int b : kBpwF64)
            if (fits(b)) break;
    }
    return p;
}

namespace {
// Holds `blocks` of a device's compute units from a launch until its end.
struct CuHold {
    CuBudget &bud;
    const int blocks;
    CuHold(int device, int blocks_, int cus) : bud(g_budget[device]), blocks(blocks_) { bud.acquire(blocks, cus); }
    ~CuHold() { bud.release(blocks); }
};
// the state to the host; waits also after an error, for what runs
hipError_t finish_resident(hipStream_t st, const SolveState *state, SolveState *h_state) {
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(h_state, state, sizeof(SolveState), hipMemcpyDeviceToHost, st);
    const hipError_t e2 = hipStreamSynchronize(st);
    return e != hipSuccess ? e : e2;
}
}  // namespace

ResidentPlan resident_csr_plan(int64_t rows, int64_t longest, int device, int cus) {
    ResidentPlan p;
    if (device < 0 || device >= kMaxDevices || rows < 1 || longest > kCsrW) return p;
    const int cap = cus < kMaxWg ? cus : kMaxWg;
    // three rows fill a wave's registers (four spill 105 of them)
    for (int rpt = 1; rpt <= 3; ++rpt)
        if (rows <= (int64_t)cap * RT * rpt) {
            p.bpw = rpt;
            p.blocks = (int)((rows + RT * rpt - 1) / (RT * rpt));
            break;
        }
    return p;
}

hipError_t resident_csr(hipStream_t st, const ResidentPlan &p, const CsrOp &op, const double *rhs, const double *sig,
                        double *x, double *pub, unsigned long long *slots, SolveState *state, SolveState *h_state,
                        double tol_rel, int64_t max_iter, double wait, int device, int cus) {
    const uint32_t limit = (uint32_t)(wait * kTicksPerSecond);
    const CuHold hold(device, p.blocks, cus);
    hipLaunchKernelGGL(k_resident_begin, dim3((kSlotWords + 255) / 256), dim3(256), 0, st, state, slots);
    auto kern = p.bpw == 1 ? k_csr_resident<1> : p.bpw == 2 ? k_csr_resident<2> : k_csr_resident<3>;
    hipLaunchKernelGGL(kern, dim3(p.blocks), dim3(RT), 0, st, op, rhs, sig, x, pub, slots, state, tol_rel, max_iter,
                       limit);
    return finish_resident(st, state, h_state);
}

template <class T>
hipError_t resident_cg(hipStream_t st, const ResidentPlan &p, const BrickOp<T> &op, const T *rhs, const double *sig,
                       T *x, T *faces, unsigned long long *slots, SolveState *state, SolveState *h_state,
                       double tol_rel, int64_t max_iter, double wait, int device, int cus) {
    const uint32_t limit = (uint32_t)(wait * kTicksPerSecond);
    const CuHold hold(device, p.blocks, cus);
    hipLaunchKernelGGL(k_resident_begin, dim3((kSlotWords + 255) / 256), dim3(256), 0, st, state, slots);
    const bool unit = op.diag == nullptr, flat = op.bx == 64;
    if constexpr (sizeof(T) == 4) {
        if (unit && flat)
            launch_bpw<T, true, 64, false>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
        else if (unit)
            launch_bpw<T, true, 8, false>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
        else if (flat)
            launch_bpw<T, false, 64, false>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
        else
            launch_bpw<T, false, 8, false>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
    } else {
        if (unit && flat)
            launch_bpw<T, true, 64, true>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
        else if (unit)
            launch_bpw<T, true, 8, true>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
        else if (flat)
            launch_bpw<T, false, 64, false>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
        else
            launch_bpw<T, false, 8, false>(st, p, op, rhs, sig, x, faces, slots, state, tol_rel, max_iter, limit);
    }
    return finish_resident(st, state, h_state);
}

template ResidentPlan resident_plan<float>(const BrickOp<float> &, int, int);
template ResidentPlan resident_plan<double>(const BrickOp<double> &, int, int);
template hipError_t resident_cg<float>(hipStream_t, const ResidentPlan &, const BrickOp<float> &, const float *,
                                       const double *, float *, float *, unsigned long long *, SolveState *,
                                       SolveState *, double, int64_t, double, int, int);
template hipError_t resident_cg<double>(hipStream_t, const ResidentPlan &, const BrickOp<double> &, const double *,
                                        const double *, double *, double *, unsigned long long *, SolveState *,
                                        SolveState *, double, int64_t, double, int, int);

}  // namespace shk
