// Fused level kernels of the V-cycle, one instance per precision.
//
// A V-cycle level used to write an array after each operator: the iterate a
// smoothing starts from (a copy, or the correction added to the pre-smoothed
// error) with its fill, the residuum, the restricted residuum.  On the fine
// levels each of these is bound by memory, on the coarse ones by the few
// microseconds of a launch.  Here the start of a smoothing is evaluated
// while its first sweep's tile is staged in LDS, and the residuum while it is
// restricted, so neither is stored.  Every value is produced by the
// expressions of the separate kernels (stencil.h) in their order, so the
// results are the same.
//
// The fill is resolved beforehand into one source cell and sign per cell
// (MgFill): with its chains of patches and faces followed in the kernel, the
// few workgroups next to an obstacle took several times as long as the rest
// of a launch (70 us instead of 20 at 256x128x128).
#include "mg_fused.h"

#include <algorithm>

#include "stencil.h"

namespace artss {
namespace k {

namespace {

constexpr int kTX = 64;  // cells of a tile along x: one wavefront
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kItemLanes = 8;  // lanes (and words) per fill item

struct Dims {
    int N[3], n[3];
};
inline Dims dims_of(const LevelDesc &L) { return {{L.N[0], L.N[1], L.N[2]}, {L.n[0], L.n[1], L.n[2]}}; }

__device__ __forceinline__ unsigned at(const Dims &L, int i, int j, int k) {
    return static_cast<unsigned>(i) +
           static_cast<unsigned>(L.N[0]) * (static_cast<unsigned>(j) + static_cast<unsigned>(L.N[1]) * static_cast<unsigned>(k));
}
__device__ __forceinline__ void cell_of(const Dims &L, unsigned u, int &i, int &j, int &k) {
    const unsigned Nx = static_cast<unsigned>(L.N[0]), Ny = static_cast<unsigned>(L.N[1]), row = u / Nx;
    i = static_cast<int>(u - row * Nx);
    k = static_cast<int>(row / Ny);
    j = static_cast<int>(row - static_cast<unsigned>(k) * Ny);
}
__device__ __forceinline__ unsigned source_of(int e) { return static_cast<unsigned>(e < 0 ? -e : e) - 1u; }

template <typename T>
struct Sweep {
    T ax, ay, az, beta, dsign, w;
};
template <typename T>
inline Sweep<T> sweep_of(const MgSweep &c) {
    return {static_cast<T>(c.ax), static_cast<T>(c.ay), static_cast<T>(c.az),
            static_cast<T>(c.beta), static_cast<T>(c.dsign), static_cast<T>(c.w)};
}

// Obstacle boxes that the region of a tile is tested against
struct Boxes {
    int n;
    Box box[kMaxObstacles];
};
inline Boxes boxes_of(const LevelDesc &L) {
    Boxes b;
    b.n = L.n_obst;
    std::copy(L.obst, L.obst + L.n_obst, b.box);
    return b;
}
__device__ __forceinline__ bool meets(const Boxes &b, int x0, int x1, int y0, int y1, int z0, int z1) {
    bool hit = false;
    for (int m = 0; m < b.n; m++) {
        const int a0 = b.box[m].lo[0], a1 = b.box[m].hi[0], b0 = b.box[m].lo[1], b1 = b.box[m].hi[1],
                  c0 = b.box[m].lo[2], c1 = b.box[m].hi[2];
        hit = hit | ((x1 >= a0) & (x0 <= a1) & (y1 >= b0) & (y0 <= b1) & (z1 >= c0) & (z0 <= c1));
    }
    return hit;
}

// The level of an iterate and, for a correction, the coarse level
template <typename T, typename TB, typename Tc>
struct Start {
    Dims L, Lc;
    const int32_t *src_of;     // MgFill of the level
    const int32_t *coarse_of;  // ... and of the coarse level
    const T *x;
    const TB *b;
    const Tc *coarse;
};

// The four values of one coarse plane a prolongation reads, and the value it
// gives from the plane of the fine cell's parent and the plane on its side.
// FP64 keeps the operand order of dev::prolong_t (the reference's).  The FP32
// iterate (the preconditioner's) takes the weights (3, 1) / 4 axis by axis,
// with one sum per plane that two fine planes share: 5 instead of 16
// operations per cell, and no larger rounding error.
template <typename T, typename Tc, bool SEPARABLE>
struct CoarsePlane {
    Tc c, x, y, xy;
    __device__ __forceinline__ void set(Tc c_, Tc x_, Tc y_, Tc xy_) {
        c = c_, x = x_, y = y_, xy = xy_;
    }
    __device__ __forceinline__ T with(const CoarsePlane &z) const {
        return static_cast<T>(static_cast<Tc>(0.015625) *
                              (27 * c + 9 * x + 9 * y + 9 * z.c + 3 * xy + 3 * z.x + 3 * z.y + z.xy));
    }
};
template <typename T, typename Tc>
struct CoarsePlane<T, Tc, true> {
    Tc sum;
    __device__ __forceinline__ void set(Tc c, Tc x, Tc y, Tc xy) { sum = 3 * (3 * c + x) + (3 * y + xy); }
    __device__ __forceinline__ T with(const CoarsePlane &z) const {
        return static_cast<T>(static_cast<Tc>(0.015625) * (3 * sum + z.sum));
    }
};

// The iterate a smoothing starts from at a cell the fill does not write, in
// two halves: its loads, which have no branch around them so that those of
// several cells are in flight together, and its value.  Where the cell lies
// under a coarse obstacle no correction is added (coarse_of not nullptr).
template <typename T, typename TB, typename Tc, bool FROM_B, bool COARSE>
struct IterateAt {
    T v;         // x, or b
    Tc c[8];     // the coarse cell and its neighbours toward the fine cell's side, x fastest
    bool reach;  // a correction is added

    __device__ __forceinline__ void load(const Start<T, TB, Tc> &S, int i, int j, int k) {
        const unsigned idx = at(S.L, i, j, k);
        if (FROM_B) v = static_cast<T>(S.b[idx]);
        else v = S.x[idx];
        if (!COARSE) return;
        const int ci = (i + 1) / 2, cj = (j + 1) / 2, ck = (k + 1) / 2;
        reach = (ci >= 1) & (cj >= 1) & (ck >= 1) & (ci <= S.Lc.n[0]) & (cj <= S.Lc.n[1]) & (ck <= S.Lc.n[2]);
        // (clamped: read where the prolongation does not reach as well)
        const int nj = S.Lc.N[0], nk = S.Lc.N[0] * S.Lc.N[1];
        const int oi = (i & 1) ? -1 : 1, oj = (j & 1) ? -nj : nj, ok = (k & 1) ? -nk : nk;
        const int n = static_cast<int>(
            at(S.Lc, min(max(ci, 1), S.Lc.n[0]), min(max(cj, 1), S.Lc.n[1]), min(max(ck, 1), S.Lc.n[2])));
        reach = reach & (S.coarse_of[n] == n + 1);
        c[0] = S.coarse[n];
        c[1] = S.coarse[n + oi];
        c[2] = S.coarse[n + oj];
        c[3] = S.coarse[n + oi + oj];
        c[4] = S.coarse[n + ok];
        c[5] = S.coarse[n + oi + ok];
        c[6] = S.coarse[n + oj + ok];
        c[7] = S.coarse[n + oi + oj + ok];
    }
    __device__ __forceinline__ T value(const Sweep<T> &s) const {
        T r = v;
        if (FROM_B) r = s.w * (s.beta * (s.dsign * r));
        if (COARSE) {
            CoarsePlane<T, Tc, sizeof(T) == 4> p, q;
            p.set(c[0], c[1], c[2], c[3]);
            q.set(c[4], c[5], c[6], c[7]);
            r = r + (reach ? p.with(q) : T(0));
        }
        return r;
    }
};

// the face ghosts set from inner fluid cell (i, j, k) of value v
template <typename T>
struct FaceGhosts {
    int active;
    int target[6];
    T sign[6];
};
template <typename T>
inline FaceGhosts<T> ghosts_of(const MgFill &F) {
    FaceGhosts<T> g;
    g.active = F.active;
    for (int p = 0; p < 6; p++) {
        g.target[p] = F.target[p];
        g.sign[p] = static_cast<T>(F.sign[p]);
    }
    return g;
}
template <typename T>
__device__ __forceinline__ void write_ghosts(const Dims &L, const FaceGhosts<T> &G, T *dst, int i, int j, int k, T v) {
    if (!G.active) return;
    if (i == G.target[0]) dst[at(L, 0, j, k)] = G.sign[0] * v + T(0);
    if (i == G.target[1]) dst[at(L, L.N[0] - 1, j, k)] = G.sign[1] * v + T(0);
    if (j == G.target[2]) dst[at(L, i, 0, k)] = G.sign[2] * v + T(0);
    if (j == G.target[3]) dst[at(L, i, L.N[1] - 1, k)] = G.sign[3] * v + T(0);
    if (k == G.target[4]) dst[at(L, i, j, 0)] = G.sign[4] * v + T(0);
    if (k == G.target[5]) dst[at(L, i, j, L.N[2] - 1)] = G.sign[5] * v + T(0);
}

// k_smooth_start: a workgroup stages the iterate on a kTX x TY x TZ tile and
// its six faces in LDS and after one barrier sweeps the tile.  A wavefront
// stages columns along z of 64 cells of a row, so that the coarse planes of a
// correction are read and summed once per column; next to the domain's faces
// a column takes the values of the row or plane its ghosts mirror.  Tiles
// where the fill or the correction is less regular (MAPPED: an obstacle or
// coarse obstacle, a periodic face along z, an odd number of cells) look
// every cell's source up first, U rows per wavefront and step.  Fill items
// run in extra workgroups: eight lanes evaluate the iterate on an item's
// source cell and its six neighbours.
template <typename T, typename TB, typename Tc, bool FROM_B, bool COARSE, int TY, int TZ>
__global__ void __launch_bounds__(kThreads)
    k_smooth_start(Start<T, TB, Tc> S, Boxes boxes, FaceGhosts<T> G, const int32_t *__restrict__ items, int n_items,
                   int gx, int gy, int gz, Sweep<T> c, T *__restrict__ dst) {
    using Iterate = IterateAt<T, TB, Tc, FROM_B, COARSE>;
    __shared__ T tile[TZ + 2][TY + 2][kTX + 4];
    const Dims &L = S.L;
    const unsigned main = static_cast<unsigned>(gx) * static_cast<unsigned>(gy) * static_cast<unsigned>(gz);
    if (blockIdx.x >= main) {
        const int u = static_cast<int>(blockIdx.x - main) * kThreads + static_cast<int>(threadIdx.x);
        if (u / kItemLanes >= n_items) return;
        const int l = static_cast<int>(threadIdx.x) & (kItemLanes - 1);
        const int lane0 = (static_cast<int>(threadIdx.x) & 63) - l;
        const int e = items[u];
        T v = T(0), rhs = T(0);
        if (l < 7 && e != 0) {
            int i, j, k;
            cell_of(L, source_of(e), i, j, k);
            Iterate it;
            it.load(S, i, j, k);
            if (l == 0) rhs = static_cast<T>(S.b[source_of(e)]);
            v = it.value(c);
            if (l > 0) v = (e < 0 ? T(-1) : T(1)) * v + T(0);
        }
        const T xp = __shfl(v, lane0 + 1, 64), xm = __shfl(v, lane0 + 2, 64), yp = __shfl(v, lane0 + 3, 64),
                ym = __shfl(v, lane0 + 4, 64), zp = __shfl(v, lane0 + 5, 64), zm = __shfl(v, lane0 + 6, 64);
        const int to = __shfl(e, lane0 + 7, 64);
        if (l != 0 || to == 0) return;
        if (e > 0) {
            const T out_h = c.beta * (c.dsign * rhs + c.ax * (xp + xm) + c.ay * (yp + ym) + c.az * (zp + zm));
            v = (1 - c.w) * v + c.w * out_h;
        } else if (FROM_B && !COARSE) {
            v = T(0);
        }
        dst[source_of(to)] = (to < 0 ? T(-1) : T(1)) * v + T(0);
        return;
    }
    // (contiguous runs of tiles per XCD: neighbours share its L2)
    const unsigned id = blockIdx.x, per = main / 8u;
    const unsigned nid = id < per * 8u ? (id % 8u) * per + id / 8u : id;
    const int bx = static_cast<int>(nid % static_cast<unsigned>(gx));
    const int by = static_cast<int>(nid / static_cast<unsigned>(gx) % static_cast<unsigned>(gy));
    const int bz = static_cast<int>(nid / static_cast<unsigned>(gx * gy));
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int i0 = 1 + bx * kTX, j0 = 1 + by * TY, k0 = 1 + bz * TZ;
    const int i1 = min(i0 + kTX - 1, L.n[0]), j1 = min(j0 + TY - 1, L.n[1]), k1 = min(k0 + TZ - 1, L.n[2]);
    const int i = i0 + lane, ic = min(i, i1);
    const int h = COARSE ? 1 : 0;
    const bool lo0 = i0 == 1, hi0 = i1 == L.n[0], lo1 = j0 == 1, hi1 = j1 == L.n[1], lo2 = k0 == 1, hi2 = k1 == L.n[2];
    const bool shell = lo0 | hi0 | lo1 | hi1 | lo2 | hi2;
    bool mapped = meets(boxes, (i0 - 1 + h) >> h, (i1 + 1 + h) >> h, (j0 - 1 + h) >> h, (j1 + 1 + h) >> h,
                        (k0 - 1 + h) >> h, (k1 + 1 + h) >> h);
    mapped = mapped | (shell & (G.active == 0)) | (lo2 & (G.target[4] != 1)) | (hi2 & (G.target[5] != L.n[2]));
    // (a periodic face may meet an obstacle on the far side)
    mapped = mapped | ((boxes.n > 0) & ((lo0 & (G.target[0] != 1)) | (hi0 & (G.target[1] != L.n[0])) |
                                        (lo1 & (G.target[2] != 1)) | (hi1 & (G.target[3] != L.n[1]))));
    if (COARSE)
        mapped = mapped | (hi0 & (L.n[0] != 2 * S.Lc.n[0])) | (hi1 & (L.n[1] != 2 * S.Lc.n[1])) |
                 (hi2 & (L.n[2] != 2 * S.Lc.n[2]));
    constexpr int kRows = (TY + 2) * (TZ + 2), kOwn = TY * TZ / kWaves;
    static_assert(TZ % 2 == 0 && TY * TZ % kWaves == 0, "tile");
    static_assert(2 * TY * TZ <= kThreads, "one column cell per thread");
    // the right-hand side of the sweep
    T rhs[kOwn];
    int own[kOwn];
#pragma unroll
    for (int u = 0; u < kOwn; u++) {
        const int r = wave + u * kWaves;
        const unsigned idx = at(L, ic, min(j0 + r % TY, j1), min(k0 + r / TY, k1));
        rhs[u] = static_cast<T>(S.b[idx]);
        own[u] = mapped ? S.src_of[idx] : static_cast<int>(idx) + 1;
    }
    // the cells left and right of the tile
    const int side = static_cast<int>(threadIdx.x) & 1, cy = (static_cast<int>(threadIdx.x) >> 1) % TY,
              cz = (static_cast<int>(threadIdx.x) >> 1) / TY;
    const bool column = static_cast<int>(threadIdx.x) < 2 * TY * TZ && j0 + cy <= j1 && k0 + cz <= k1;
    Iterate col;
    int ce = 0;
    if (column) {
        int ci = side ? i1 + 1 : i0 - 1, cj = j0 + cy, ck = k0 + cz;
        const unsigned idx = at(L, ci, cj, ck);
        ce = S.src_of[idx];
        cell_of(L, ce != 0 ? source_of(ce) : idx, ci, cj, ck);
        col.load(S, ci, cj, ck);
    }
    if (mapped) {
        constexpr int U = sizeof(T) == 4 ? 6 : 3;
        auto row = [&](int r, int &y, int &z, int &j, int &k) {
            r = min(r, kRows - 1);
            y = r % (TY + 2);
            z = r / (TY + 2);
            j = min(j0 + y - 1, j1 + 1);
            k = min(k0 + z - 1, k1 + 1);
        };
#pragma unroll 1
        for (int r0 = wave; r0 < kRows; r0 += kWaves * U) {
            Iterate it[U];
            int e[U];
            unsigned idx[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                int y, z, j, k;
                row(r0 + u * kWaves, y, z, j, k);
                idx[u] = at(L, ic, j, k);
                e[u] = S.src_of[idx[u]];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                int si, sj, sk;
                cell_of(L, e[u] != 0 ? source_of(e[u]) : idx[u], si, sj, sk);
                it[u].load(S, si, sj, sk);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                int y, z, j, k;
                row(r0 + u * kWaves, y, z, j, k);
                T v = it[u].value(c);
                if (FROM_B && !COARSE && e[u] == 0) v = T(0);
                if (e[u] < 0) v = -v;
                if (i <= i1) tile[z][y][lane + 1] = v;
            }
        }
    } else {
        const unsigned plane = static_cast<unsigned>(L.N[0]) * static_cast<unsigned>(L.N[1]);
        const int ci = (ic + 1) / 2, oi = (ic & 1) ? -1 : 1;
        const int cplane = S.Lc.N[0] * S.Lc.N[1];
#pragma unroll 1
        for (int y = wave; y < TY + 2; y += kWaves) {
            int j = min(j0 + y - 1, j1 + 1);
            T gs = T(1);
            if (j == 0) {
                gs = G.sign[2];
                j = G.target[2];
            } else if (j == L.N[1] - 1) {
                gs = G.sign[3];
                j = G.target[3];
            }
            T v[TZ + 2];
            const unsigned base = at(L, ic, j, 0);
#pragma unroll
            for (int z = 0; z < TZ + 2; z++) {
                const unsigned idx = base + plane * static_cast<unsigned>(min(k0 + z - 1, L.N[2] - 1));
                v[z] = FROM_B ? static_cast<T>(S.b[idx]) : S.x[FROM_B ? 0 : idx];
            }
            CoarsePlane<T, Tc, sizeof(T) == 4> q[TZ / 2 + 2];
            if (COARSE) {
                // (k0 is odd: the planes (k0 - 1) / 2 ... of the coarse level)
                const int cn = static_cast<int>(at(S.Lc, ci, (j + 1) / 2, 0)), oj = (j & 1) ? -S.Lc.N[0] : S.Lc.N[0];
#pragma unroll
                for (int p = 0; p < TZ / 2 + 2; p++) {
                    const int n = cn + cplane * min((k0 - 1) / 2 + p, S.Lc.N[2] - 1);
                    q[p].set(S.coarse[n], S.coarse[n + oi], S.coarse[n + oj], S.coarse[n + oi + oj]);
                }
            }
#pragma unroll
            for (int z = 0; z < TZ + 2; z++) {
                if (FROM_B) v[z] = c.w * (c.beta * (c.dsign * v[z]));
                // even k: the parent's upper neighbour, odd k: its lower one
                if (COARSE) v[z] = v[z] + ((z & 1) ? q[(z + 1) / 2].with(q[(z - 1) / 2]) : q[z / 2].with(q[z / 2 + 1]));
            }
            if (k0 == 1) v[0] = G.sign[4] * v[1];
#pragma unroll
            for (int z = 1; z < TZ + 2; z++)
                if (k0 + z - 1 == L.N[2] - 1) v[z] = G.sign[5] * v[z - 1];
            if (i <= i1) {
#pragma unroll
                for (int z = 0; z < TZ + 2; z++) tile[z][y][lane + 1] = gs * v[z];
            }
        }
    }
    if (column) {
        T v = col.value(c);
        if (FROM_B && !COARSE && ce == 0) v = T(0);
        if (ce < 0) v = -v;
        tile[cz + 1][cy + 1][side ? i1 - i0 + 2 : 0] = v;
    }
    __syncthreads();
    if (i > i1) return;
#pragma unroll
    for (int u = 0; u < kOwn; u++) {
        const int r = wave + u * kWaves, y = r % TY, z = r / TY;
        const int j = j0 + y, k = k0 + z;
        if (j > j1 || k > k1) continue;
        const unsigned idx = at(L, i, j, k);
        const T v0 = tile[z + 1][y + 1][lane + 1];
        const T out_h = c.beta * (c.dsign * rhs[u] +
                                  c.ax * (tile[z + 1][y + 1][lane + 2] + tile[z + 1][y + 1][lane]) +
                                  c.ay * (tile[z + 1][y + 2][lane + 1] + tile[z + 1][y][lane + 1]) +
                                  c.az * (tile[z + 2][y + 1][lane + 1] + tile[z][y + 1][lane + 1]));
        const T v = (1 - c.w) * v0 + c.w * out_h;
        if (!mapped) {
            dst[idx] = v;
            if (shell) write_ghosts(L, G, dst, i, j, k, v);
        } else if (own[u] == static_cast<int>(idx) + 1) {
            dst[idx] = v;
            write_ghosts(L, G, dst, i, j, k, v);
        } else if (own[u] == 0) {
            dst[idx] = v0;
        }
    }
}

// 1 / h^2 of the fine level, formed as dev::laplace_t forms them
template <typename T>
struct LapCoef {
    T x, y, z;
};

// k_residuum_restrict: one thread per coarse cell evaluates the residuum of
// its eight fine cells from the 32 values they read (an obstacle grows when
// it is coarsened, so a coarse fluid cell has fluid children only).  FROM_B:
// the values next to the shell or an obstacle are looked up.  Bound by
// memory where the level is large: at 256x128x128 in FP32 14 us (of reading b
// once, 7) in place of 15 for the sweep from zero, 13 for the residuum and 9
// for the restriction; on small levels one launch (5 us) in place of two.
template <typename T, typename TB, typename Tout, bool FROM_B>
__global__ void __launch_bounds__(kThreads)
    k_residuum_restrict(Dims Lc, Dims Lf, Boxes boxes, const int32_t *__restrict__ src_of, Sweep<T> c, LapCoef<T> h,
                        Tout *__restrict__ out, Tout *__restrict__ err, const T *__restrict__ x,
                        const TB *__restrict__ b) {
    const unsigned gx = gridDim.x, gy = gridDim.y;
    const unsigned id = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), per = gx * gy * gridDim.z / 8u;
    const unsigned nid = id < per * 8u ? (id % 8u) * per + id / 8u : id;
    const int o = err != nullptr ? 0 : 1;
    const int i = o + static_cast<int>(nid % gx) * 64 + static_cast<int>(threadIdx.x);
    const int j = o + static_cast<int>(nid / gx % gy) * kWaves + static_cast<int>(threadIdx.y);
    const int k = o + static_cast<int>(nid / (gx * gy));
    if (i >= Lc.N[0] - o || j >= Lc.N[1] - o) return;
    const unsigned cidx = at(Lc, i, j, k);
    if (err != nullptr) err[cidx] = Tout(0);
    if (i < 1 || j < 1 || k < 1 || i > Lc.n[0] || j > Lc.n[1] || k > Lc.n[2]) return;
    if (meets(boxes, i, i, j, j, k, k)) return;
    // fine coordinates 2 i - 2 .. 2 i + 1 per axis, from the corner cell's index
    const unsigned corner = at(Lf, 2 * i - 2, 2 * j - 2, 2 * k - 2);
    const unsigned nj = static_cast<unsigned>(Lf.N[0]), nk = nj * static_cast<unsigned>(Lf.N[1]);
    auto outer = [](int e, int f, int g) { return (e == 0 || e == 3) + (f == 0 || f == 3) + (g == 0 || g == 3); };
    T v[4][4][4], bv[2][2][2];
    int m[4][4][4];
    bool near = false;
    if (FROM_B) {
        near = (i == 1) | (j == 1) | (k == 1) | (2 * i + 1 > Lf.n[0]) | (2 * j + 1 > Lf.n[1]) | (2 * k + 1 > Lf.n[2]) |
               meets(boxes, i - 1, i + 1, j - 1, j + 1, k - 1, k + 1);
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int f = 0; f < 4; f++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (outer(e, f, g) == 1) m[g][f][e] = static_cast<int>(corner + e + nj * f + nk * g) + 1;
        if (near) {
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int f = 0; f < 4; f++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (outer(e, f, g) == 1) m[g][f][e] = src_of[corner + e + nj * f + nk * g];
        }
    }
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
        for (int f = 0; f < 4; f++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (outer(e, f, g) > 1) continue;
                const bool own = outer(e, f, g) == 0;
                const unsigned idx = corner + e + nj * f + nk * g;
                if (own) bv[g - 1][f - 1][e - 1] = static_cast<T>(b[idx]);
                if (!FROM_B) {
                    v[g][f][e] = x[idx];
                } else if (own) {
                    v[g][f][e] = c.w * (c.beta * (c.dsign * bv[g - 1][f - 1][e - 1]));
                } else {
                    const int n = m[g][f][e];
                    T value = c.w * (c.beta * (c.dsign * static_cast<T>(b[n != 0 ? source_of(n) : idx])));
                    if (n == 0) value = T(0);
                    v[g][f][e] = n < 0 ? -value : value;
                }
            }
    T sum = T(0);
#pragma unroll
    for (int n = 0; n < 8; n++) {
        const int e = 1 + (n & 1), f = 1 + ((n >> 1) & 1), g = 1 + (n >> 2);
        const T x0 = v[g][f][e];
        const T lap = (h.x * (v[g][f][e - 1] - 2 * x0 + v[g][f][e + 1]) +
                       h.y * (v[g][f - 1][e] - 2 * x0 + v[g][f + 1][e]) +
                       h.z * (v[g - 1][f][e] - 2 * x0 + v[g + 1][f][e]));
        const T res = bv[g - 1][f - 1][e - 1] - lap;
        sum = n == 0 ? res : sum + res;
    }
    out[cidx] = static_cast<Tout>(static_cast<T>(0.125) * sum);
}

// ---- MgFill tables, three launches: each reads what the one before wrote
__global__ void k_map_cells(LevelDesc L, int32_t *__restrict__ map) {
    const long long n = blockIdx.x * 256LL + threadIdx.x;
    if (n >= L.size) return;
    const unsigned u = static_cast<unsigned>(n), Nx = static_cast<unsigned>(L.N[0]), Ny = static_cast<unsigned>(L.N[1]);
    const int i = static_cast<int>(u % Nx), j = static_cast<int>((u / Nx) % Ny), k = static_cast<int>(u / (Nx * Ny));
    const bool fluid = i >= 1 && j >= 1 && k >= 1 && i <= L.n[0] && j <= L.n[1] && k <= L.n[2] && !in_obstacle(L, i, j, k);
    map[n] = fluid ? static_cast<int32_t>(n + 1) : 0;
}
__global__ void k_map_faces(BCView V, int32_t *__restrict__ map) {
    const long long t = blockIdx.x * 256LL + threadIdx.x;
    if (t >= V.n_faces) return;
    const FaceEntry e = V.faces[t];
    const FaceParam q = V.params[e.param];
    if (!q.active) return;
    const int32_t src = static_cast<int32_t>(e.idx) + e.ref + 1;
    map[e.idx] = q.sign < 0.0 ? -src : src;
}
__device__ __forceinline__ double ghost_sign(const LevelDesc &L, const DomainBC &bc, long long i, long long j,
                                             long long k) {
    return dev::ghost_chain<double>(L, bc, i, j, k, 1.0);  // the values are zero
}
__global__ void k_map_ghosts(LevelDesc L, BCView V, int32_t *__restrict__ map) {
    const long long t = blockIdx.x * 256LL + threadIdx.x;
    long long i, j, k;
    if (t >= V.n_ghosts || !dev::ghost_coords(L, t, i, j, k)) return;
    // (the source is a cell the fill does not write or an obstacle face)
    const long long src = dev::ghost_source(L, V.bc, i, j, k);
    const int32_t e = dev::written(V, src) ? map[src] : static_cast<int32_t>(src + 1);
    map[dev::lin(L, i, j, k)] = ghost_sign(L, V.bc, i, j, k) < 0.0 ? -e : e;
}
__global__ void k_map_items(LevelDesc L, BCView V, const int32_t *__restrict__ map, int32_t *__restrict__ items,
                            int n_items) {
    const long long q = blockIdx.x * 256LL + threadIdx.x;
    if (q >= n_items) return;
    long long t = q, cell = -1;
    if (t < V.n_faces) {
        const FaceEntry e = V.faces[t];
        long long i = e.idx % L.N[0], j = (e.idx / L.N[0]) % L.N[1], k = e.idx / (static_cast<long long>(L.N[0]) * L.N[1]);
        const bool shell = i == 0 || j == 0 || k == 0 || i == L.N[0] - 1 || j == L.N[1] - 1 || k == L.N[2] - 1;
        // (a face on the ghost layer is overwritten by the ghosts)
        if (!(shell && V.n_ghosts != 0)) cell = e.idx;
    } else if ((t -= V.n_faces) < V.n_rest) {
        cell = V.rest[t];
    } else if ((t -= V.n_rest) < V.n_deps) {
        cell = V.deps[t].idx;
    } else {
        long long i, j, k;
        if (dev::ghost_coords(L, t - V.n_deps, i, j, k) && !dev::written(V, dev::lin(L, i, j, k))) cell = dev::lin(L, i, j, k);
    }
    int32_t *out = items + 8 * q;
    for (int a = 0; a < 8; a++) out[a] = 0;
    if (cell < 0) return;
    const int32_t e = map[cell];
    const long long src = e == 0 ? cell : (e < 0 ? -static_cast<long long>(e) : e) - 1;
    const bool fluid = map[src] == static_cast<int32_t>(src + 1);
    const long long nj = L.N[0], nk = nj * L.N[1];
    out[0] = static_cast<int32_t>(fluid ? src + 1 : -(src + 1));
    if (fluid) {
        out[1] = map[src + 1];
        out[2] = map[src - 1];
        out[3] = map[src + nj];
        out[4] = map[src - nj];
        out[5] = map[src + nk];
        out[6] = map[src - nk];
    }
    out[7] = static_cast<int32_t>(e < 0 ? -(cell + 1) : cell + 1);
}

template <typename T, typename TB, typename Tc, bool FROM_B, bool COARSE, int TY, int TZ>
void launch_start(hipStream_t s, const Start<T, TB, Tc> &S, const Boxes &boxes, const MgFill &F, const MgSweep &c,
                  T *dst) {
    const int gx = (S.L.n[0] + kTX - 1) / kTX, gy = (S.L.n[1] + TY - 1) / TY, gz = (S.L.n[2] + TZ - 1) / TZ;
    const long long blocks =
        static_cast<long long>(gx) * gy * gz + (static_cast<long long>(F.n_items) * kItemLanes + kThreads - 1) / kThreads;
    k_smooth_start<T, TB, Tc, FROM_B, COARSE, TY, TZ><<<static_cast<unsigned>(blocks), kThreads, 0, s>>>(
        S, boxes, ghosts_of<T>(F), F.items, F.n_items, gx, gy, gz, sweep_of<T>(c), dst);
}

template <typename T, typename TB, typename Tc, bool FROM_B, bool COARSE>
void pick_start(hipStream_t s, const Start<T, TB, Tc> &S, const Boxes &boxes, const MgFill &F, const MgSweep &c, T *dst) {
    const long long rows = static_cast<long long>((S.L.n[0] + kTX - 1) / kTX) * S.L.n[1] * S.L.n[2];
    // Large levels are bound by issue and by the cells staged twice: deeper
    // tiles (256x128x128 in FP32: 29 us, with the small tile 44; 128^3 in
    // FP64: 21 against 23 us).  Small ones are bound by the chain of loads of
    // a wavefront and by the workgroups there are: one column of six cells
    // per wavefront (128x64x64: 7 us, with a 64x8x8 tile 19).
    if (rows >= 16384)
        launch_start<T, TB, Tc, FROM_B, COARSE, sizeof(T) == 4 ? 6 : 2, sizeof(T) == 4 ? 4 : 8>(s, S, boxes, F, c, dst);
    else
        launch_start<T, TB, Tc, FROM_B, COARSE, 2, 4>(s, S, boxes, F, c, dst);
}

}  // namespace

void build_mg_fill(hipStream_t s, const LevelDesc &L, const BCView &V, int32_t *map, int32_t *items, int n_items) {
    auto blocks = [](long long n) { return static_cast<unsigned>((n + 255) / 256); };
    k_map_cells<<<blocks(L.size), 256, 0, s>>>(L, map);
    if (V.n_faces > 0) k_map_faces<<<blocks(V.n_faces), 256, 0, s>>>(V, map);
    if (V.n_ghosts > 0) k_map_ghosts<<<blocks(V.n_ghosts), 256, 0, s>>>(L, V, map);
    if (n_items > 0) k_map_items<<<blocks(n_items), 256, 0, s>>>(L, V, map, items, n_items);
}
template <typename T, typename TB>
void smooth_first(hipStream_t s, const LevelDesc &L, const MgFill &F, const MgSweep &c, T *dst, const T *x,
                  const TB *b) {
    const Start<T, TB, T> S{dims_of(L), dims_of(L), F.src_of, nullptr, x, b, nullptr};
    if (x == nullptr) pick_start<T, TB, T, true, false>(s, S, boxes_of(L), F, c, dst);
    else pick_start<T, TB, T, false, false>(s, S, boxes_of(L), F, c, dst);
}
template void smooth_first<double, double>(hipStream_t, const LevelDesc &, const MgFill &, const MgSweep &, double *,
                                           const double *, const double *);
template void smooth_first<float, double>(hipStream_t, const LevelDesc &, const MgFill &, const MgSweep &, float *,
                                          const float *, const double *);
template void smooth_first<float, float>(hipStream_t, const LevelDesc &, const MgFill &, const MgSweep &, float *,
                                         const float *, const float *);
template <typename T, typename TB, typename Tc>
void smooth_corrected(hipStream_t s, const LevelDesc &L, const MgFill &F, const MgSweep &c, T *dst, const T *x,
                      const TB *b, const LevelDesc &Lc, const MgFill &Fc, const Tc *coarse) {
    const Start<T, TB, Tc> S{dims_of(L), dims_of(Lc), F.src_of, Fc.src_of, x, b, coarse};
    if constexpr (sizeof(T) == sizeof(float)) {
        if (x == nullptr) {
            pick_start<T, TB, Tc, true, true>(s, S, boxes_of(Lc), F, c, dst);
            return;
        }
    }
    pick_start<T, TB, Tc, false, true>(s, S, boxes_of(Lc), F, c, dst);
}
#define ARTSS_CORRECTED(T, TB, Tc)                                                                                 \
    template void smooth_corrected<T, TB, Tc>(hipStream_t, const LevelDesc &, const MgFill &, const MgSweep &, T *, \
                                              const T *, const TB *, const LevelDesc &, const MgFill &, const Tc *);
ARTSS_CORRECTED(double, double, double)
ARTSS_CORRECTED(float, double, float)
ARTSS_CORRECTED(float, double, double)
ARTSS_CORRECTED(float, float, float)
ARTSS_CORRECTED(float, float, double)
#undef ARTSS_CORRECTED

template <typename T, typename TB, typename Tout>
void residuum_restrict(hipStream_t s, const LevelDesc &Lc, const LevelDesc &Lf, const MgFill &F, const MgSweep &c,
                       Tout *out, Tout *err, const T *x, const TB *b) {
    const LapCoef<T> h{static_cast<T>(1. / (Lf.h[0] * Lf.h[0])), static_cast<T>(1. / (Lf.h[1] * Lf.h[1])),
                       static_cast<T>(1. / (Lf.h[2] * Lf.h[2]))};
    const int *n = err != nullptr ? Lc.N : Lc.n;
    const dim3 g((n[0] + 63) / 64, (n[1] + kWaves - 1) / kWaves, n[2]), t(64, kWaves);
    if constexpr (sizeof(T) == sizeof(float)) {
        if (x == nullptr) {
            k_residuum_restrict<T, TB, Tout, true><<<g, t, 0, s>>>(dims_of(Lc), dims_of(Lf), boxes_of(Lc), F.src_of,
                                                                   sweep_of<T>(c), h, out, err, x, b);
            return;
        }
    }
    k_residuum_restrict<T, TB, Tout, false><<<g, t, 0, s>>>(dims_of(Lc), dims_of(Lf), boxes_of(Lc), F.src_of,
                                                            sweep_of<T>(c), h, out, err, x, b);
}
#define ARTSS_RESTRICT(T, TB, Tout)                                                                         \
    template void residuum_restrict<T, TB, Tout>(hipStream_t, const LevelDesc &, const LevelDesc &,         \
                                                 const MgFill &, const MgSweep &, Tout *, Tout *, const T *, \
                                                 const TB *);
ARTSS_RESTRICT(double, double, double)
ARTSS_RESTRICT(float, double, float)
ARTSS_RESTRICT(float, double, double)
ARTSS_RESTRICT(float, float, float)
ARTSS_RESTRICT(float, float, double)
#undef ARTSS_RESTRICT

}  // namespace k
}  // namespace artss
