// The small levels of a reference-hierarchy V-cycle, two launches around the
// coarsest solve (gfx950).
//
// Below 16^3 cells a level's kernels hold a few microseconds of launch and
// memory latency each for almost no work, and a V-cycle visits every such
// level with eight of them (smoothing, residual, restriction, tau,
// prolongation, smoothing). k_tail_down takes the cycle from the first level
// of at most kTailCells cells down to the coarsest level's right-hand side
// in one workgroup, k_tail_up from the coarsest solution back. Each lane
// owns up to four cells of a level, two of each colour, and keeps their
// rows and right-hand sides in registers; the solution stays in LDS, one
// array for the level at hand, and so do the face conductances of rows in
// exact arithmetic (three arrays: a cell's - faces are its neighbours' +
// faces). The rows come formed from k_tail_rows, which runs once per set of
// coefficients and boundary codes: the per-level kernels form them, with six
// divisions each, in every pass, and in these kernels 16 waves on one CU
// took 26 us a visit for it. What bounds a launch is latency: per colour
// pass an LDS round trip, the row's chain, a division and a barrier; per
// level a round trip to memory for its rows. So index divisions are float
// products, the prolongation reads a ghosted array of coarse corrections
// whose ghosts their owners wrote, and a level of one wave's cells takes no
// barriers.
// Measured per V-cycle, 16^3 and 8^3 above a 64-cell coarsest grid, exact rows
// with convection: 27 us down and 21 us up, where the per-level kernels took
// 14 launches and about 125 us; 16^3 to 2^3, explicit rows in FP64: 41 and 26
// us against 33 launches and about 170 us. (Rows formed in these kernels: 44
// and 51 us; coarse corrections looked up with the ghost rule's branches per
// neighbour: 16 us a level going up.)
//
// The arithmetic is the per-level kernels': in exact arithmetic every
// operation in the reference's order (row(), k_restrict_fas, k_tau,
// k_prolong1_correct, with a row's terms as k_bottom_wave forms them), so
// the cycle is the same bit for bit; fast rows from coefficients and
// explicit rows as k_sweep_fast's.
#pragma once

#include "mps3d_bottom.h"
#include "mps3d_sweep.h"

namespace mps {

constexpr int kTailCells = 4096;    // the first level's most cells
constexpr int kTailThreads = 1024;
constexpr int kTailLev = 6;         // levels including the coarsest
constexpr int kTailSlots = kTailCells / 2 / kTailThreads;   // cells of one colour per lane
constexpr int kTailGhosted = 2304;  // ghosted cells of any level below the first

template <typename T>
struct TailLevels {
    Lev<T> L[kTailLev];
    T *u[kTailLev], *uold[kTailLev], *b[kTailLev];
    T *rows[kTailLev];            // k_tail_rows' output (rows from coefficients)
    const T *face[kTailLev][6];   // BC faces for the prolongation's ghost rule (nullable = 0)
    int nlev, nu;
};

// q / d for 0 <= q < 2^20 and a small d: the product's relative error (2^-22)
// is below the distance 1 / 2d of (q + 1/2) / d from the next integer
struct SmallDiv {
    int d;
    float inv;
    __device__ __forceinline__ explicit SmallDiv(int d_) : d(d_), inv(1.0f / (float)d_) {}
    __device__ __forceinline__ int operator()(int q) const { return (int)(((float)q + 0.5f) * inv); }
};

// one owned cell: its place, its row and its right-hand side
struct TailPlace {
    int q;         // natural index in the level (-1: none)
    int ex;        // bit f: face f has a neighbour
    int c;         // index in the ghosted arrays
};
template <typename T, int NK, int NV>
struct TailCell : TailPlace {
    T dg, b;
    T k[NK], v[NV];
};

template <typename T, int OP, bool VEL, bool LIN>
struct Tail {
    static constexpr bool GL = !LIN;   // exact rows: face conductances in LDS
    static constexpr int NK = GL ? 1 : 6, NV = VEL ? 6 : 1;
    using Cell = TailCell<T, NK, NV>;
    struct Lds {
        T u[kTailCells + 2];
        T g[GL ? 3 : 1][GL ? kTailCells + 2 : 1];
        T e[kTailGhosted];   // ghosted coarse correction (up)
    };

    // cell t of a colour (rows of an even width: nx / 2 per row), or cell t in
    // natural order (colour < 0)
    static __device__ __forceinline__ void place(const Lev<T> &L, int t, int colour, TailPlace &C)
    {
        const int n = L.nx * L.ny * L.nz;
        C.q = -1;
        C.ex = 0;
        C.c = 0;
        if (t >= (colour < 0 ? n : n / 2)) return;
        const int w = colour < 0 ? L.nx : L.nx / 2;
        const int rw = SmallDiv(w)(t), k = SmallDiv(L.ny)(rw) + 1, j = rw - (k - 1) * L.ny + 1;
        const int p = t - rw * w;
        const int i = colour < 0 ? p + 1 : (((1 + j + k) & 1) == colour ? 1 : 2) + 2 * p;
        C.q = (i - 1) + L.nx * rw;
        C.ex = (i > 1 ? 1 : 0) | (i < L.nx ? 2 : 0) | (j > 1 ? 4 : 0) | (j < L.ny ? 8 : 0) | (k > 1 ? 16 : 0) |
               (k < L.nz ? 32 : 0);
        C.c = i + L.sy * j + (int)L.sz * k;
    }

    // the row of an owned cell (explicit rows: the level's arrays; else
    // k_tail_rows' arrays of n values: the diagonal, then the six multipliers
    // of fast rows, or the + faces' conductances and the six convective
    // multipliers of exact ones)
    static __device__ __forceinline__ void load_row(const Lev<T> &L, const T *rows, Cell &C, Lds &S, int n)
    {
        if (C.q < 0) return;
        if constexpr (OP == OP_STENCIL) {
#pragma unroll
            for (int f = 0; f < 6; ++f) C.k[f] = (C.ex >> f) & 1 ? L.st[1 + f][C.c] : T(0);
            C.dg = L.st[ST_C][C.c];
        } else {
            const T *p = rows + C.q;
            C.dg = p[0];
            if constexpr (GL) {
#pragma unroll
                for (int d = 0; d < 3; ++d) S.g[d][C.q] = p[(1 + d) * n];
                if constexpr (VEL) {
#pragma unroll
                    for (int f = 0; f < 6; ++f) C.v[f] = p[(4 + f) * n];
                }
            } else {
#pragma unroll
                for (int f = 0; f < 6; ++f) C.k[f] = p[(1 + f) * n];
            }
        }
    }

    // off-diagonal sum of an owned cell's row over the solution in LDS (entry n
    // of every array is zero: the neighbour of a face that does not exist)
    static __device__ __forceinline__ T offdiag(const Lev<T> &L, const Cell &C, const Lds &S, int n)
    {
        const int of[6] = {-1, 1, -L.nx, L.nx, -L.nx * L.ny, L.nx * L.ny};
        const T ab[3] = {L.ax, L.ay, L.az};
        int nb[6];
        T un[6], kf[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            nb[f] = (C.ex >> f) & 1 ? C.q + of[f] : n;
            un[f] = S.u[nb[f]];
            if constexpr (GL) kf[f] = -S.g[f / 2][(f & 1) ? C.q : nb[f]];
            else kf[f] = C.k[f];
        }
        T o = T(0);
        if constexpr (LIN) {
#pragma clang fp contract(fast)
#pragma unroll
            for (int f = 0; f < 6; ++f) o = o + kf[f] * un[f];
        } else {
#pragma unroll
            for (int f = 0; f < 6; ++f) {
                T t = un[f] * kf[f] * ab[f / 2];
                if constexpr (VEL) t = t + C.v[f] * un[f] * ab[f / 2];
                o = o + t;
            }
        }
        return o;
    }

    static __device__ __forceinline__ T update(const Lev<T> &L, const Cell &C, T o, T old)
    {
        T v;
        if constexpr (LIN && OP != OP_STENCIL) v = (C.b - o) * fast_rcp(C.dg);
        else v = gs_update(L, C.b, o, C.dg);
        if (LIN && L.omega != T(1)) v = old + L.omega * (v - old);
        return v;
    }

    // nu red-black sweeps; cells[0..kTailSlots) are red, the others black.
    // Ends (and, for nu > 0, every pass ends) with the new values visible.
    static __device__ __forceinline__ void smooth(const Lev<T> &L, const Cell *cells, Lds &S, int n, int nu)
    {
        const bool solo = n <= 128;   // both colours within the first wave
        for (int s = 0; s < nu; ++s) {
#pragma unroll
            for (int colour = 0; colour < 2; ++colour) {
                // (a colour's cells read only the other colour and themselves,
                // so each is stored as soon as it is formed; one cell at a
                // time: more in flight spills)
#pragma unroll
                for (int p = 0; p < kTailSlots; ++p) {
                    const Cell &C = cells[colour * kTailSlots + p];
                    if (C.q >= 0) S.u[C.q] = update(L, C, offdiag(L, C, S, n), LIN ? S.u[C.q] : T(0));
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (solo) wave_fence();
                else __syncthreads();
            }
        }
        if (solo) __syncthreads();
    }
};

constexpr int kTailRowArrays = 10;   // per cell, at most (exact rows with convection)

// the rows of the levels k_tail_down and k_tail_up hold (blockIdx.y), one
// thread per cell: the diagonal as row() forms it, and each face's
// multiplier(s) of the neighbour value as k_bottom_wave's
template <typename T, bool VEL, bool REAC, bool LIN>
__global__ void __launch_bounds__(kBlock) k_tail_rows(TailLevels<T> A)
{
    const Lev<T> &L = A.L[blockIdx.y];
    const int n = L.nx * L.ny * L.nz, q = blockIdx.x * kBlock + threadIdx.x;
    if (q >= n) return;
    const int rw = q / L.nx, i = q - rw * L.nx + 1, k = rw / L.ny + 1, j = rw - (k - 1) * L.ny + 1;
    const long long c = (long long)i + (long long)L.sy * j + L.sz * k;
    const bool ex[6] = {i > 1, i < L.nx, j > 1, j < L.ny, k > 1, k < L.nz};
    const long long st[3] = {1, L.sy, L.sz};
    T *const p = A.rows[blockIdx.y] + q;
    const T Dc = L.D[c];
    if constexpr (LIN) {
#pragma clang fp contract(fast)
        const T hf[3] = {L.hx, L.hy, L.hz}, gf[3] = {L.gx, L.gy, L.gz};
        T d = T(0);
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const T w = ex[f] ? (L.D[(f & 1) ? c + st[f / 2] : c - st[f / 2]] + Dc) * hf[f / 2] : T(0);
            p[(1 + f) * n] = -w;
            d += w;
            if (!ex[f] && L.bc[f] == BC_DIRC) d += Dc * gf[f / 2];
        }
        if (REAC) d -= L.reac[c];
        p[0] = d + L.dtinv;
    } else {
        T dg, of;
        row<T, OP_REF, VEL, REAC>(L, L.D, i, j, k, c, dg, of);   // (the diagonal does not read u)
        p[0] = dg;
        const T h[3] = {L.dx, L.dy, L.dz};
        const T *v3[3] = {L.vx, L.vy, L.vz};
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const int d = f / 2;
            const long long o = (f & 1) ? c + st[d] : c - st[d];
            if (f & 1) p[(1 + d) * n] = ex[f] ? (T(0.5) * (Dc + L.D[o])) / h[d] : T(0);
            if constexpr (VEL) {
                // the upwind cell of a face is the left one where vh > 0
                const T vh = T(0.5) * ((f & 1) ? v3[d][c] + v3[d][o] : v3[d][o] + v3[d][c]);
                p[(4 + f) * n] = (ex[f] && (vh > T(0)) == !(f & 1)) ? ((f & 1) ? vh : -vh) : T(0);
            }
        }
    }
}

template <typename T, int OP, bool VEL, bool LIN>
__global__ void __launch_bounds__(kTailThreads) k_tail_down(TailLevels<T> A)
{
    using K = Tail<T, OP, VEL, LIN>;
    using Cell = typename K::Cell;
    __shared__ typename K::Lds S;
    const int tid = threadIdx.x;
    constexpr int NC = 2 * kTailSlots;
    Cell cells[NC];
    // the first level's solution and right-hand side
#pragma unroll
    for (int p = 0; p < NC; ++p) {
        K::place(A.L[0], tid + kTailThreads * (p % kTailSlots), p < kTailSlots ? 1 : 0, cells[p]);
        if (cells[p].q >= 0) {
            S.u[cells[p].q] = A.u[0][cells[p].c];
            cells[p].b = A.b[0][cells[p].c];
        }
    }
    for (int l = 0;; ++l) {
        const Lev<T> &L = A.L[l];
        const int n = L.nx * L.ny * L.nz;
#pragma unroll
        for (int p = 0; p < NC; ++p) K::load_row(L, A.rows[l], cells[p], S, n);
        if (tid == 0) {
            S.u[n] = T(0);
            if constexpr (K::GL)
                for (int d = 0; d < 3; ++d) S.g[d][n] = T(0);
        }
        __syncthreads();
        if (l > 0) {
            // tau (k_tau): b = A(R u) + R r
#pragma unroll
            for (int p = 0; p < NC; p += kTailSlots) {
                Cell &C = cells[p];
                if (C.q < 0) continue;
                const T uo = S.u[C.q];
                const T of = K::offdiag(L, C, S, n);
                C.b = (C.dg * uo + of) + C.b;
                A.b[l][C.c] = C.b;
                A.uold[l][C.c] = uo;
                if (l == A.nlev - 1) A.u[l][C.c] = uo;
            }
            if (l == A.nlev - 1) return;
            __syncthreads();
        }
        K::smooth(L, cells, S, n, A.nu);
        // residual, and the coarse cells' sums of the solution (k_restrict_fas)
        T r[NC];
#pragma unroll
        for (int p = 0; p < NC; ++p) {
            const Cell &C = cells[p];
            r[p] = T(0);
            if (C.q < 0) continue;
            const T u = S.u[C.q], of = K::offdiag(L, C, S, n);
            r[p] = C.b - (C.dg * u + of);
            A.u[l][C.c] = u;
            __builtin_amdgcn_sched_barrier(0);
        }
        const Lev<T> &Lc = A.L[l + 1];
        const bool last = l + 1 == A.nlev - 1;
        const int sy = L.nx, sz = L.nx * L.ny;
        const int o[8] = {0, 1, sy, sy + 1, sz, sz + 1, sz + sy, sz + sy + 1};
        // (the next level has at most kTailCells / 8 cells: slot 0 of a
        // colour, or one cell in natural order on the coarsest level)
        TailPlace next[2];
        int f0[2];
        T us[2], nb[2];
        auto gather = [&](int x) {
            T s = T(0);
#pragma unroll
            for (int w = 0; w < 8; ++w) s = s + S.u[f0[x] + o[w]];
            return T(1.0 / 8.0) * s;
        };
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            K::place(Lc, (last && x) ? kTailCells : tid, last ? -1 : 1 - x, next[x]);
            f0[x] = 0;
            us[x] = nb[x] = T(0);
            if (next[x].q >= 0) {
                const int rw = SmallDiv(Lc.nx)(next[x].q), i = next[x].q - rw * Lc.nx, k = SmallDiv(Lc.ny)(rw),
                          j = rw - k * Lc.ny;
                f0[x] = 2 * i + sy * 2 * j + sz * 2 * k;
                us[x] = gather(x);
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < NC; ++p)
            if (cells[p].q >= 0) S.u[cells[p].q] = r[p];
        __syncthreads();
#pragma unroll
        for (int x = 0; x < 2; ++x)
            if (next[x].q >= 0) nb[x] = gather(x);
        __syncthreads();
#pragma unroll
        for (int p = 0; p < NC; ++p) cells[p].q = -1;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            static_cast<TailPlace &>(cells[x * kTailSlots]) = next[x];
            cells[x * kTailSlots].b = nb[x];
            if (next[x].q >= 0) S.u[next[x].q] = us[x];
        }
    }
}

template <typename T, int OP, bool VEL, bool LIN>
__global__ void __launch_bounds__(kTailThreads) k_tail_up(TailLevels<T> A)
{
    using K = Tail<T, OP, VEL, LIN>;
    using Cell = typename K::Cell;
    __shared__ typename K::Lds S;
    const int tid = threadIdx.x;
    constexpr int NC = 2 * kTailSlots;
    // a coarse cell's correction (error_2h = unew - uold) into the ghosted
    // array, with the ghosts of the boundary faces it touches: the rule of
    // err_at (update_boundary_ghostvalues on both)
    auto put = [&](int l, const TailPlace &C, T un, T uo) {
        const Lev<T> &L = A.L[l];
        const int st[3] = {1, L.sy, (int)L.sz};
        const T *F[6];
        bool dirc[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) {   // (uniform loads together, before the faces' branches)
            F[f] = A.face[l][f];
            dirc[f] = L.bc[f] == BC_DIRC;
        }
        S.e[C.c] = un - uo;
        if (C.ex == 63) return;
        const int rw = SmallDiv(L.nx)(C.q), i = C.q - rw * L.nx, k = SmallDiv(L.ny)(rw), j = rw - k * L.ny;
        const int fi[3] = {j + L.ny * k, i + L.nx * k, i + L.nx * j};
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            if ((C.ex >> f) & 1) continue;
            T e = un - uo;
            if (dirc[f]) {
                const T g2 = F[f] ? T(2) * F[f][fi[f / 2]] : T(0);
                e = (g2 - un) - (g2 - uo);
            }
            S.e[(f & 1) ? C.c + st[f / 2] : C.c - st[f / 2]] = e;
        }
    };
    {
        const int lb = A.nlev - 1;
        TailPlace C;
        K::place(A.L[lb], tid, -1, C);
        if (C.q >= 0) put(lb, C, A.u[lb][C.c], A.uold[lb][C.c]);
    }
    for (int l = A.nlev - 2; l >= 0; --l) {
        const Lev<T> &L = A.L[l], &Lc = A.L[l + 1];
        const int n = L.nx * L.ny * L.nz;
        Cell cells[NC];
        T u[NC], uo[2];
#pragma unroll
        for (int p = 0; p < NC; ++p) {
            K::place(L, tid + kTailThreads * (p % kTailSlots), p < kTailSlots ? 1 : 0, cells[p]);
            u[p] = T(0);
            if (cells[p].q >= 0) {
                u[p] = A.u[l][cells[p].c];
                cells[p].b = A.b[l][cells[p].c];
            }
            // (levels below the first: slot 0 of a colour)
            if (p % kTailSlots == 0) uo[p / kTailSlots] = l > 0 && cells[p].q >= 0 ? A.uold[l][cells[p].c] : T(0);
            K::load_row(L, A.rows[l], cells[p], S, n);
        }
        if (tid == 0) {
            S.u[n] = T(0);
            if constexpr (K::GL)
                for (int d = 0; d < 3; ++d) S.g[d][n] = T(0);
        }
        __syncthreads();
        // prolongation1 and correction (k_prolong1_correct), per fine cell
        const int cy = Lc.sy, cz = (int)Lc.sz;
#pragma unroll
        for (int p = 0; p < NC; ++p) {
            const Cell &C = cells[p];
            if (C.q < 0) continue;
            const int rw = SmallDiv(L.nx)(C.q), i = C.q - rw * L.nx, k = SmallDiv(L.ny)(rw), j = rw - k * L.ny;
            const T *E = S.e + ((i / 2 + 1) + cy * (j / 2 + 1) + cz * (k / 2 + 1));
            const T e = E[0];
            const T sx = T(0.5) * (E[1] - E[-1]);
            const T sy = T(0.5) * (E[cy] - E[-cy]);
            const T sz = T(0.5) * (E[cz] - E[-cz]);
            T t = (i & 1) ? sx : -sx;
            t = (j & 1) ? t + sy : t - sy;
            t = (k & 1) ? t + sz : t - sz;
            S.u[C.q] = u[p] + (e + T(0.25) * t);
        }
        __syncthreads();
        K::smooth(L, cells, S, n, A.nu);
        if (l == 0) {
#pragma unroll
            for (int p = 0; p < NC; ++p)
                if (cells[p].q >= 0) A.u[0][cells[p].c] = S.u[cells[p].q];
        } else {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const Cell &C = cells[x * kTailSlots];
                if (C.q >= 0) put(l, C, S.u[C.q], uo[x]);
            }
        }
    }
}

}  // namespace mps
