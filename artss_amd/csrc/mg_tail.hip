// Single-workgroup kernel for the coarse end of a multigrid V-cycle.
//
// The levels it covers hold at most a few ten thousand cells, so one
// workgroup of 1024 threads (16 wavefronts on one CU) walks each of them in
// a strided loop and a workgroup barrier separates consecutive operators.
// Every operator is the one VCycleMG applies at that point
// (VCycleMG.cpp:215-288, :299-308, :562-798), evaluated with the same
// per-cell functions as the multi-workgroup kernels (stencil.h), so the
// result is bit-identical to issuing those kernels one by one; only the
// coarse solve's residual sum is formed in this kernel's own fixed order.
#include "mg_plan.h"
#include "mg_tail.h"
#include "stencil.h"

#include <mutex>

namespace artss {
namespace {

using dev::lin;

// Each thread handles kBatch cells per pass: their loads are all issued
// before the first store, so a pass costs one memory round trip instead of
// kBatch of them.
constexpr int kBatch = 4;
constexpr int kStride = kTailThreads * kBatch;

struct Cell {
    int idx;   // linear index in the level array (levels here are small)
    bool on;   // an inner (fluid) cell
};

// inner-box cell number t (x fastest) of level L
__device__ inline Cell box_cell(const LevelDesc &L, int t, int n) {
    Cell c{0, false};
    if (t >= n) return c;
    const int nx = L.n[0], ny = L.n[1];
    const int i = 1 + t % nx, r = t / nx;
    const int j = 1 + r % ny, k = 1 + r / ny;
    c.on = !in_obstacle(L, i, j, k);
    c.idx = i + L.N[0] * (j + L.N[1] * k);
    return c;
}

__device__ inline int box_cells(const LevelDesc &L) { return L.n[0] * L.n[1] * L.n[2]; }

// DomainController::apply_boundary: obstacle faces wave by wave, then ghosts
__device__ __forceinline__ void t_bc(const TailLevel &T, double *f) {
    for (int w = 0; w < T.n_waves; w++) {
        const int e0 = static_cast<int>(T.wave_start[w]), e1 = static_cast<int>(T.wave_start[w + 1]);
        for (int e = e0 + threadIdx.x; e < e1; e += kTailThreads) dev::face_write(T.faces[e], T.params, f);
        __syncthreads();
    }
    if (T.bc.active) {
        const int n = static_cast<int>(dev::ghost_count(T.L));
        for (int t = threadIdx.x; t < n; t += kTailThreads) dev::domain_ghost(T.L, T.bc, f, t);
        __syncthreads();
    }
}

__device__ __forceinline__ void t_copy(double *__restrict__ dst, const double *__restrict__ src, int n) {
    for (int base = threadIdx.x; base < n; base += kStride) {
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int t = base + u * kTailThreads;
            if (t < n) v[u] = src[t];
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int t = base + u * kTailThreads;
            if (t < n) dst[t] = v[u];
        }
    }
    __syncthreads();
}

__device__ __forceinline__ void t_fill(double *dst, double v, int n) {
    for (int t = threadIdx.x; t < n; t += kTailThreads) dst[t] = v;
    __syncthreads();
}

__device__ __forceinline__ void t_add(double *__restrict__ dst, const double *__restrict__ src, int n) {
    for (int base = threadIdx.x; base < n; base += kStride) {
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int t = base + u * kTailThreads;
            if (t < n) v[u] = dst[t] + src[t];
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int t = base + u * kTailThreads;
            if (t < n) dst[t] = v[u];
        }
    }
    __syncthreads();
}

__device__ __forceinline__ void t_jacobi(const TailLevel &T, const TailPlan &P, double *__restrict__ out,
                         const double *__restrict__ in, const double *__restrict__ b) {
    const int n = box_cells(T.L);
    for (int base = threadIdx.x; base < n; base += kStride) {
        Cell c[kBatch];
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            c[u] = box_cell(T.L, base + u * kTailThreads, n);
            if (c[u].on) v[u] = dev::jacobi_mg(T.L, T.ax, T.ay, T.az, T.beta, P.dsign, P.w, in, b, c[u].idx);
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (c[u].on) out[c[u].idx] = v[u];
    }
    __syncthreads();
}

// one color, in place: cells of a color read only cells of the other color
__device__ __forceinline__ void t_cgs_color(const TailLevel &T, const TailPlan &P, int color, double *out, const double *b) {
    const int n = box_cells(T.L);
    const int nx = T.L.n[0], ny = T.L.n[1];
    for (int base = threadIdx.x; base < n; base += kStride) {
        Cell c[kBatch];
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int t = base + u * kTailThreads;
            c[u] = box_cell(T.L, t, n);
            if (c[u].on) {
                const int i = 1 + t % nx, r = t / nx;
                const int j = 1 + r % ny, k = 1 + r / ny;
                c[u].on = ((i + j + k) & 1) == color;
            }
            if (c[u].on) v[u] = dev::cgs_mg(T.L, T.ax, T.ay, T.az, T.beta, P.dsign, P.w, out, b, c[u].idx);
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (c[u].on) out[c[u].idx] = v[u];
    }
    __syncthreads();
}

__device__ __forceinline__ void t_residuum(const TailLevel &T, double *__restrict__ out, const double *__restrict__ x,
                           const double *__restrict__ b) {
    const int n = box_cells(T.L);
    for (int base = threadIdx.x; base < n; base += kStride) {
        Cell c[kBatch];
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            c[u] = box_cell(T.L, base + u * kTailThreads, n);
            if (c[u].on) v[u] = b[c[u].idx] - dev::laplace(T.L, x, c[u].idx);
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (c[u].on) out[c[u].idx] = v[u];
    }
    __syncthreads();
}

// ||b - lap x||_2 over the inner cells, same value in every thread
__device__ __forceinline__ double t_residual(const TailLevel &T, const double *__restrict__ x, const double *__restrict__ b,
                             double *red) {
    const int n = box_cells(T.L);
    double sq = 0.0;
    for (int base = threadIdx.x; base < n; base += kStride) {
        Cell c[kBatch];
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            c[u] = box_cell(T.L, base + u * kTailThreads, n);
            v[u] = c[u].on ? b[c[u].idx] - dev::laplace(T.L, x, c[u].idx) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++) sq += v[u] * v[u];
    }
    for (int off = 32; off > 0; off >>= 1) sq += __shfl_down(sq, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kTailThreads / 64; w++) s += red[w];
        red[kTailThreads / 64] = sqrt(s);
    }
    __syncthreads();
    const double r = red[kTailThreads / 64];
    __syncthreads();
    return r;
}

__device__ __forceinline__ void t_restrict(const TailLevel &Tc, const TailLevel &Tf, double *__restrict__ out,
                           const double *__restrict__ in) {
    const int n = box_cells(Tc.L);
    const int nx = Tc.L.n[0], ny = Tc.L.n[1];
    for (int base = threadIdx.x; base < n; base += kStride) {
        Cell c[kBatch];
        double v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int t = base + u * kTailThreads;
            c[u] = box_cell(Tc.L, t, n);
            if (c[u].on) {
                const int i = 1 + t % nx, r = t / nx;
                const int j = 1 + r % ny, k = 1 + r / ny;
                v[u] = dev::restrict_cell(Tf.L, in, i, j, k);
            }
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (c[u].on) out[c[u].idx] = v[u];
    }
    __syncthreads();
}

__device__ __forceinline__ void t_prolongate(const TailLevel &Tc, const TailLevel &Tf, double *__restrict__ out,
                             const double *__restrict__ in) {
    const int n = box_cells(Tc.L);
    const int nx = Tc.L.n[0], ny = Tc.L.n[1];
    for (int t = threadIdx.x; t < n; t += kTailThreads) {
        const Cell c = box_cell(Tc.L, t, n);
        if (!c.on) continue;
        const int i = 1 + t % nx, r = t / nx;
        const int j = 1 + r % ny, k = 1 + r / ny;
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = dev::prolong_value(Tc.L, in, c.idx, q);
#pragma unroll
        for (int q = 0; q < 8; q++) out[dev::prolong_target(Tf.L, i, j, k, q)] = v[q];
    }
    __syncthreads();
}

// ---- Jacobi sweeps with their state in registers
// The loop of a coarse solve is a serial chain of up to max_iter sweeps, each
// followed by its fill and its residual, on one CU: what bounds it is the
// instructions and barriers between two sweeps, not data.  So everything that
// does not change from sweep to sweep is worked out once and kept in
// registers: every thread's cells (NB of 1024 at a time; index, fluid or
// not, right-hand side), the face ghosts whose patch chain starts on them,
// and the thread's obstacle face write.  The residual of an iterate and the
// next sweep read the same seven values, so they share one pass: the next
// values are formed beside the residual and dropped when the test ends the
// loop.  A sweep then costs two workgroup barriers (three with obstacle
// faces, one without a test) instead of seven or more, and with the level
// in LDS its accesses are DS instructions instead of flat ones.
// Values are those of t_jacobi, t_bc and t_residual bit for bit: the same
// expressions, the same cells per thread and order of the sum.  Edge and
// corner ghosts, which no sweep reads, are left to the caller's fill.
// The kernel on the 20x12x8 coarse level of a 160x96x64 box (1920 cells, 100
// tested sweeps): 751 us with one pass per operator, 276 us so; on 8x8x8
// (128^3, five levels): 444 us and 175 us.

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

constexpr int kWaves = kTailThreads / 64;

// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uniform(double v) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = static_cast<unsigned>(uniform(static_cast<int>(b))),
                   hi = static_cast<unsigned>(uniform(static_cast<int>(b >> 32)));
    return __builtin_bit_cast(double, (static_cast<unsigned long long>(hi) << 32) | lo);
}

// sweeps of x_0 = out (filled; tmp a copy of it) while fewer than max_iter
// ran and, with `test`, ||b - lap x||_2 > target; x_1, x_3, .. go to out,
// x_2, x_4, .. to tmp.  relative: target is a factor on x_0's residual.
template <int NB>
__device__ __forceinline__ void t_sweeps(const TailLevel &T, const TailPlan &P, double *lds, const double *b,
                                         double *red, int max_iter, bool test, bool relative, double target) {
    const int off_tmp = uniform(T.lds_off[1]), off_out = uniform(T.lds_off[0]);
    const LevelDesc &L = T.L;
    const int n = box_cells(L);
    const int nj = uniform(L.N[0]), nk = uniform(L.N[0] * L.N[1]);
    // (read from LDS, so the compiler does not see that they are uniform)
    const double ax = uniform(T.ax), ay = uniform(T.ay), az = uniform(T.az), beta = uniform(T.beta),
                 dsign = uniform(P.dsign), w = uniform(P.w), w1 = uniform(1 - P.w);
    const double rdx2 = uniform(1. / (L.h[0] * L.h[0])), rdy2 = uniform(1. / (L.h[1] * L.h[1])),
                 rdz2 = uniform(1. / (L.h[2] * L.h[2]));
    // a cell's index (a level in LDS has fewer than 2^16 cells) and above it
    // bit 16 + p: it feeds the face ghost of patch p, bit 22: a fluid cell
    unsigned cell[NB];
    double bv[NB];
#pragma unroll
    for (int u = 0; u < NB; u++) {
        const Cell c = box_cell(L, threadIdx.x + u * kTailThreads, n);
        cell[u] = static_cast<unsigned>(nk + nj + 1);
        bv[u] = 0.0;
        if (!c.on) continue;
        const int k = c.idx / nk, r = c.idx - k * nk, j = r / nj, i = r - j * nj;
        unsigned feeds = 64u;
        if (T.bc.active)
            feeds |= (i == T.bc.target[0] ? 1u : 0u) | (i == T.bc.target[1] ? 2u : 0u) |
                     (j == T.bc.target[2] ? 4u : 0u) | (j == T.bc.target[3] ? 8u : 0u) |
                     (k == T.bc.target[4] ? 16u : 0u) | (k == T.bc.target[5] ? 32u : 0u);
        cell[u] = static_cast<unsigned>(c.idx) | (feeds << 16);
        bv[u] = b[c.idx];
    }
    const int goff[6] = {uniform(-T.bc.target[0]),      uniform(L.N[0] - 1 - T.bc.target[1]),
                         uniform(-T.bc.target[2] * nj), uniform((L.N[1] - 1 - T.bc.target[3]) * nj),
                         uniform(-T.bc.target[4] * nk), uniform((L.N[2] - 1 - T.bc.target[5]) * nk)};
    double gs[6], gv[6];
#pragma unroll
    for (int p = 0; p < 6; p++) {
        gs[p] = uniform(T.bc.sign[p]);
        gv[p] = uniform(T.bc.value[p]);
    }
    // the thread's obstacle face write
    const bool faces = T.n_waves > 0;
    int f_idx = 0, f_src = 0;
    double f_sign = 0.0, f_value = 0.0;
    bool f_on = false;
    if (faces) {
        const int e = static_cast<int>(T.wave_start[0]) + static_cast<int>(threadIdx.x);
        if (e < static_cast<int>(T.wave_start[1])) {
            const FaceEntry x = T.faces[e];
            const FaceParam q = T.params[x.param];
            f_on = q.active != 0;
            f_idx = static_cast<int>(x.idx);
            f_src = f_idx + x.ref;
            f_sign = q.sign;
            f_value = q.value;
        }
    }
    for (int it = 0; it < max_iter; it++) {
        const double *in = lds + ((it & 1) ? off_out : off_tmp);
        double *o = lds + ((it & 1) ? off_tmp : off_out);
        double v[NB], sq = 0.0;
#pragma unroll
        for (int u = 0; u < NB; u++) {
            const int i = static_cast<int>(cell[u] & 0xffffu);
            const double c = in[i], xm = in[i - 1], xp = in[i + 1], ym = in[i - nj], yp = in[i + nj],
                         zm = in[i - nk], zp = in[i + nk];
            const double r =
                bv[u] - (rdx2 * (xm - 2 * c + xp) + rdy2 * (ym - 2 * c + yp) + rdz2 * (zm - 2 * c + zp));
            sq += (cell[u] >> 16) ? r * r : 0.0;
            const double out_h = beta * (dsign * bv[u] + ax * (xp + xm) + ay * (yp + ym) + az * (zp + zm));
            v[u] = w1 * c + w * out_h;
        }
        if (test && (it > 0 || relative)) {
            double *part = red + (it & 1) * kWaves;
            sq = wave_sum(sq);
            if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sq;
            __syncthreads();
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < kWaves; q++) s += part[q];
            const double res = sqrt(s);
            if (it == 0) target = target * res;
            else if (!(res > target)) break;
        }
#pragma unroll
        for (int u = 0; u < NB; u++) {
            if (!(cell[u] >> 16)) continue;
            const int i = static_cast<int>(cell[u] & 0xffffu);
            o[i] = v[u];
            if (cell[u] & 0x3f0000u)
#pragma unroll
                for (int p = 0; p < 6; p++)
                    if (cell[u] & (0x10000u << p)) o[i + goff[p]] = gs[p] * v[u] + gv[p];
        }
        __syncthreads();
        if (faces) {
            if (f_on) o[f_idx] = f_sign * o[f_src] + f_value;
            __syncthreads();
        }
    }
    __syncthreads();
}

// Levels the register sweeps take: in LDS with at most NB cells per thread; obstacle
// faces in one wave of at most one write per thread (one wave reads no cell
// that a face write changes); and no fluid cell may read a ghost whose chain
// starts off the fluid, which with a ghost's source beside it (Dirichlet,
// Neumann) holds by itself and with a periodic patch needs a level without
// obstacles.
template <int NB>
__device__ __forceinline__ bool t_sweeps_fit(const TailLevel &T) {
    if (T.lds_off[0] < 0 || T.lds_off[1] < 0 || box_cells(T.L) > NB * kTailThreads || T.n_waves > 1) return false;
    if (T.n_waves == 1 && T.wave_start[1] - T.wave_start[0] > kTailThreads) return false;
    if (T.L.n_obst == 0 || !T.bc.active) return true;
    bool beside = true;
    for (int a = 0; a < 3; a++) beside = beside && T.bc.target[2 * a] == 1 && T.bc.target[2 * a + 1] == T.L.N[a] - 2;
    return beside;
}

// The smoothing (test = false) and the coarse solve with weighted Jacobi on
// levels the register sweeps do not take: max_iter sweeps, or until the
// residual meets the target.
__device__ __forceinline__ void t_sweeps_plain(const TailLevel &T, const TailPlan &P, double *out, double *tmp,
                                               const double *b, double *red, int max_iter, bool test, bool relative,
                                               double target) {
    double *o = out, *s = tmp;
    if (relative) target = target * t_residual(T, o, b, red);
    for (int it = 0; it < max_iter; it++) {
        t_jacobi(T, P, o, s, b);
        t_bc(T, o);
        if (test && !(t_residual(T, o, b, red) > target)) break;
        double *x = o;
        o = s;
        s = x;
    }
}

// VCycleMG.cpp:583-615 (test = false) and :617-683
__device__ __forceinline__ void t_sweeps_cgs(const TailLevel &T, const TailPlan &P, double *out, const double *b,
                                             double *red, int max_iter, bool test, bool relative, double target) {
    if (relative) target = target * t_residual(T, out, b, red);
    for (int it = 0; it < max_iter; it++) {
        t_cgs_color(T, P, 0, out, b);
        t_cgs_color(T, P, 1, out, b);
        t_bc(T, out);
        if (test && !(t_residual(T, out, b, red) > target)) break;
    }
}

// VCycleMG::Smooth :299-308 (solve = false) or VCycleMG::Solve :562-581.
//
// Jacobi (VCycleMG.cpp:685-798): the reference swaps the two buffers after
// every sweep and once more after an odd count, so `out` always ends in its
// own buffer, which holds the last sweep for an odd count and the one before
// it for an even count.  The last sweep of an even smoothing is never read
// and is skipped.
//
// The coarse solve's stopping test: coarse_tol == 0, the reference's
// res > tol (absolute); coarse_tol > 0, res > coarse_tol * (the residual of
// the starting iterate), a reduction independent of the right-hand side's
// scale; coarse_tol < 0, no test (max_iter sweeps, no residual computed).
template <int NB>
__device__ __forceinline__ void t_relax(const TailLevel &T, const TailPlan &P, double *lds, double *out, double *tmp,
                                        const double *b, double *red, bool solve, double coarse_tol) {
    solve = solve && !P.solve_smooths;
    const bool test = solve && coarse_tol >= 0.0, relative = solve && coarse_tol > 0.0;
    const double target = relative ? coarse_tol : P.tol;
    int n = solve ? P.max_iter : P.n_relax;
    t_bc(T, out);
    // Smooth's own fill and the smoother's: the second matters only where
    // the fill is not idempotent
    if (!solve && T.n_waves > 1) t_bc(T, out);
    if (P.cgs) {
        t_sweeps_cgs(T, P, out, b, red, n, test, relative, target);
        return;
    }
    if (!solve && n % 2 == 0 && n > 0) n--;
    t_copy(tmp, out, static_cast<int>(T.L.size));
    if (!t_sweeps_fit<NB>(T)) {
        t_sweeps_plain(T, P, out, tmp, b, red, n, test, relative, target);
        return;
    }
    t_sweeps<NB>(T, P, lds, b, red, n, test, relative, target);
    t_bc(T, out);
}

// NB: cells per thread of the register sweeps (1 or 2, one instance each:
// both in one kernel spill, and so does a third with four cells)
template <int NB>
__global__ void __launch_bounds__(kTailThreads) k_mg_tail(const TailPlan *__restrict__ plan, const double *b_first,
                                                           int max_iter, int n_relax, double w, int skip_dead,
                                                           double coarse_tol) {
    __shared__ TailPlan P;
    __shared__ double red[2 * (kTailThreads / 64) + 1];
    extern __shared__ double lds[];
    {
        const unsigned long long *src = reinterpret_cast<const unsigned long long *>(plan);
        unsigned long long *dst = reinterpret_cast<unsigned long long *>(&P);
        constexpr int words = sizeof(TailPlan) / sizeof(unsigned long long);
        for (int t = threadIdx.x; t < words; t += kTailThreads) dst[t] = src[t];
        __syncthreads();
        if (max_iter > 0 && threadIdx.x == 0) P.max_iter = max_iter;
        if (n_relax > 0 && threadIdx.x == 0) P.n_relax = n_relax;
        if (w > 0.0 && threadIdx.x == 0) P.w = w;
        __syncthreads();
    }
    const int f = P.first, Lm = P.last;
    // Level arrays placed in LDS start as the HBM arrays they stand for: zero
    // wherever no operator writes them (every array is zero-initialised and
    // those cells are never written), the first level's error and
    // right-hand side copied in.  Only the first level's error leaves.
    if (P.lds_doubles > 0) {
        for (int t = threadIdx.x; t < P.lds_doubles; t += kTailThreads) lds[t] = 0.0;
        if (threadIdx.x == 0) {
            for (int l = 0; l <= Lm - f; l++) {
                TailLevel &T = P.lv[l];
                double **ptr[5] = {&T.err1, &T.tmp, &T.res0, &T.res1, &T.err0};
                for (int a = 0; a < 5; a++)
                    if (T.lds_off[a] >= 0) *ptr[a] = lds + T.lds_off[a];
            }
        }
        __syncthreads();
        if (P.lv[0].lds_off[0] >= 0) {
            t_copy(P.lv[0].err1, P.io_err1, static_cast<int>(P.lv[0].L.size));
            t_copy(P.lv[0].res1, b_first, static_cast<int>(P.lv[0].L.size));
            b_first = P.lv[0].res1;
        }
    }
    // descent (VCycleMG.cpp:228-252), then ascent (:255-281): one loop, so
    // that the relaxation's code stands once
    const int depth = Lm - f;
    for (int q = 0; q < 2 * depth; q++) {
        const bool down = q < depth;
        const int l = down ? q : 2 * depth - 1 - q;  // level - f
        const TailLevel &T = P.lv[l];
        const TailLevel &Tc = P.lv[l + 1];
        const double *rhs = l == 0 ? b_first : T.res1;
        // the coarsest level only ever holds a zero error (VCycleMG.cpp:228-282
        // restrict to it, then prolongate its zero back): skipped on request
        const bool skip = skip_dead && l + 1 == depth;
        if (!down && !skip) {
            t_prolongate(Tc, T, T.err0, Tc.err1);
            t_bc(T, T.err0);
            t_add(T.err1, T.err0, static_cast<int>(T.L.size));
        }
        t_relax<NB>(T, P, lds, T.err1, T.tmp, rhs, red, !down && l + 1 == depth, coarse_tol);
        if (down && !skip) {
            t_residuum(T, T.res0, T.err1, rhs);
            t_bc(T, T.res0);
            t_restrict(Tc, T, Tc.res1, T.res0);
            t_bc(Tc, Tc.res1);
            t_fill(Tc.err1, 0.0, static_cast<int>(Tc.L.size));
        }
    }
    if (P.lv[0].lds_off[0] >= 0) t_copy(P.io_err1, P.lv[0].err1, static_cast<int>(P.lv[0].L.size));
}

}  // namespace

int mg_tail_lds_limit() {
    int dev = 0, bytes = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 0;
    const int static_bytes = static_cast<int>(sizeof(TailPlan)) + 1024;
    return bytes > static_bytes ? bytes - static_bytes : 0;
}

// The attribute is per kernel function, shared by every solver in the
// process: it is only ever raised, so a smaller plan set up later does not
// invalidate the launches of a larger one.
void mg_tail_reserve_lds(int lds_bytes) {
    static std::mutex lock;
    static int reserved = 0;
    std::lock_guard<std::mutex> guard(lock);
    if (lds_bytes <= reserved) return;
    bool ok = true;
    for (const void *fn :
         {reinterpret_cast<const void *>(&k_mg_tail<1>), reinterpret_cast<const void *>(&k_mg_tail<2>)})
        ok = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) == hipSuccess && ok;
    if (ok) reserved = lds_bytes;
}

void mg_tail(hipStream_t s, const TailPlan *plan, const double *b_first, int lds_bytes, int cells, int max_iter,
             int n_relax, double w, bool skip_dead, double coarse_tol) {
    const int skip = skip_dead ? 1 : 0;
    if (cells <= kTailThreads)
        k_mg_tail<1><<<1, kTailThreads, lds_bytes, s>>>(plan, b_first, max_iter, n_relax, w, skip, coarse_tol);
    else
        k_mg_tail<2><<<1, kTailThreads, lds_bytes, s>>>(plan, b_first, max_iter, n_relax, w, skip, coarse_tol);
}

}  // namespace artss
