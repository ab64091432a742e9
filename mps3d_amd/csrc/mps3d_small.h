// The small levels of an aligned-hierarchy V-cycle in one launch (gfx950).
//
// Below about 10^3 cells a level's kernels each cost a few microseconds of
// launch and dependency latency for almost no work, and every V-cycle visits
// such a level with eight of them. k_small_cycle takes the V-cycle from one
// such level down to the dense coarsest solve and back in a single
// workgroup: it loads that level's right-hand side and the 7-point rows and
// restriction weights of every level below once, keeps all of it in LDS with
// the solutions and residuals, and writes the level's correction back.
// What bounds it is latency: the loads (one CU draws about 20 KB per
// microsecond from beyond its L2, which is what keeps 17^3 out: 275 KB of
// FP64 rows took 20 us a visit), then per colour pass an LDS round trip, the
// row's chain, a division and a barrier. So index divisions are float
// products made once per level visit, a face that does not exist reads a
// zero, and the coarsest product takes the inverse by columns (its transpose
// by rows), lanes reading consecutive values, each row's sum split over the
// lanes that the rows leave free, with the values loaded at the start.
// A lane owns one cell of each colour (index arithmetic for a second one cost
// 5 us a visit and spilled), and half the lanes, with twice the registers,
// are taken where they are enough: fewer waves at each barrier.
// Measured per visit: 17.6 us for 9^3 and 5^3 in FP64, 23.5 us for the same
// levels of 257^3 in FP32 with over-relaxed sweeps, 25.3 us for 13 x 9 x 11
// over 7 x 5 x 6 (210 rows of the inverse) in FP32. A solve at 33^3 with
// the explicit levels launched one kernel a phase took 1202 us, with this
// 1013 us; a drift-diffusion gradient step at 65^3 2369 us, with this 2003.
//
// The phases -- red-black smoothing, residual, full weighting, trilinear
// prolongation-correction -- are the per-level kernels' for explicit rows.
#pragma once

#include "mps3d_tail.h"

namespace mps {

constexpr int kSmallThreads = 1024;       // lanes, one cell of a colour each
constexpr int kSmallHalf = 512;            // where these are enough, half of them
constexpr int kSmallLev = 5;               // levels including the coarsest
constexpr int kSmallBytes = 144 * 1024;    // LDS of the levels' arrays

template <typename T>
struct SmallLevels {
    Lev<T> L[kSmallLev];
    AlignedW W[kSmallLev];      // W[q]: full-weighting weights onto level q
    T omega[kSmallLev];         // over-relaxation of the level's sweeps
    T *u0;                      // the first level's correction
    const T *b0;                // and its right-hand side
    const double *invT;         // transposed dense inverse of the coarsest operator
    int nlev, nu1, nu2;
    int zero;                   // the first level starts from zero (u0 is not read)
};

// LDS bytes of a level: u (and a zero), b, diagonal, six multipliers, and
// the weights onto it
template <typename T>
__host__ __device__ inline int small_level_bytes(int nx, int ny, int nz)
{
    const int words = 9 * nx * ny * nz + 1;
    return (words * (int)sizeof(T) + 7) / 8 * 8 + 3 * (nx + ny + nz) * 8;
}

template <typename T>
struct SmallView {
    int nx, ny, nz, n;
    T *u, *b, *dg, *k;          // k: six arrays of n
    double *wx, *wy, *wz;
};

template <typename T>
__device__ __forceinline__ SmallView<T> small_view(const SmallLevels<T> &A, unsigned char *mem, int q)
{
    int off = 0;
    for (int p = 0; p < q; ++p) off += small_level_bytes<T>(A.L[p].nx, A.L[p].ny, A.L[p].nz);
    SmallView<T> v;
    v.nx = A.L[q].nx, v.ny = A.L[q].ny, v.nz = A.L[q].nz;
    v.n = v.nx * v.ny * v.nz;
    v.wx = reinterpret_cast<double *>(mem + off);
    v.wy = v.wx + 3 * v.nx;
    v.wz = v.wy + 3 * v.ny;
    v.u = reinterpret_cast<T *>(v.wz + 3 * v.nz);
    v.b = v.u + v.n + 1;
    v.dg = v.b + v.n;
    v.k = v.dg + v.n;
    return v;
}

template <typename T>
__device__ __forceinline__ void small_ijk(const SmallView<T> &V, int q, int &i, int &j, int &k)   // 0-based
{
    const int rw = SmallDiv(V.nx)(q);
    i = q - rw * V.nx;
    k = SmallDiv(V.ny)(rw);
    j = rw - k * V.ny;
}

// cell t of a colour, numbered over rows of (nx + 1) / 2
template <typename T>
__device__ __forceinline__ TailPlace small_place(const SmallView<T> &V, int t, int colour)
{
    TailPlace C{-1, 0, 0};
    const int hx = (V.nx + 1) / 2;
    if (t >= hx * V.ny * V.nz) return C;
    const int rw = SmallDiv(hx)(t), k = SmallDiv(V.ny)(rw), j = rw - k * V.ny;
    const int i = (((1 + j + k) & 1) == colour ? 0 : 1) + 2 * (t - rw * hx);   // (i + j + k) + 3 odd: red
    if (i >= V.nx) return C;
    C.q = i + V.nx * rw;
    C.ex = (i > 0 ? 1 : 0) | (i < V.nx - 1 ? 2 : 0) | (j > 0 ? 4 : 0) | (j < V.ny - 1 ? 8 : 0) | (k > 0 ? 16 : 0) |
           (k < V.nz - 1 ? 32 : 0);
    return C;
}

template <typename T>
__device__ __forceinline__ T small_offdiag(const SmallView<T> &V, const TailPlace &C)
{
#pragma clang fp contract(fast)
    const int of[6] = {-1, 1, -V.nx, V.nx, -V.nx * V.ny, V.nx * V.ny};
    T un[6], kf[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        un[f] = V.u[(C.ex >> f) & 1 ? C.q + of[f] : V.n];
        kf[f] = V.k[f * V.n + C.q];
    }
    T o = T(0);
#pragma unroll
    for (int f = 0; f < 6; ++f) o = o + kf[f] * un[f];
    return o;
}

template <typename T>
__device__ __forceinline__ void small_smooth(const Lev<T> &L, const SmallView<T> &V, const TailPlace *cells, int nu,
                                             T omega)
{
    for (int s = 0; s < nu; ++s) {
#pragma unroll
        for (int colour = 0; colour < 2; ++colour) {
            const TailPlace &C = cells[colour];
            if (C.q >= 0) {
                T v = gs_update(L, V.b[C.q], small_offdiag(V, C), V.dg[C.q]);
                if (omega != T(1)) {
                    const T old = V.u[C.q];
                    v = old + omega * (v - old);
                }
                V.u[C.q] = v;
            }
            __syncthreads();
        }
    }
}

template <typename T, int THREADS>
__global__ void __launch_bounds__(THREADS) k_small_cycle(SmallLevels<T> A)
{
    __shared__ alignas(16) unsigned char mem[kSmallBytes];
    __shared__ double part[THREADS];   // partial sums of the coarsest product
    const int tid = threadIdx.x;
    constexpr int PRE = THREADS > kSmallHalf ? 8 : 32;   // entries of the inverse held per lane
    const int last = A.nlev - 1;
    // the coarsest product: row qb, entries hb, hb + gb, ... of its sum
    const int nb = A.L[last].nx * A.L[last].ny * A.L[last].nz, gb = THREADS / nb;
    const int hb = SmallDiv(nb)(tid), qb = tid - hb * nb;
    double inv[PRE];
#pragma unroll
    for (int p = 0; p < PRE; ++p) {
        const int e = hb + p * gb;
        inv[p] = hb < gb && e < nb ? A.invT[e * nb + qb] : 0.0;
    }
    for (int q = 0; q < A.nlev; ++q) {
        const Lev<T> &L = A.L[q];
        const SmallView<T> V = small_view(A, mem, q);
        if (q < last) {
            for (int t = tid; t < V.n; t += THREADS) {
                int i, j, k;
                small_ijk(V, t, i, j, k);
                const int c = (i + 1) + L.sy * (j + 1) + (int)L.sz * (k + 1);
                const bool ex[6] = {i > 0, i < V.nx - 1, j > 0, j < V.ny - 1, k > 0, k < V.nz - 1};
                T a[ST_N];
#pragma unroll
                for (int s = 0; s < ST_N; ++s) a[s] = L.st[s][c];
                const T b = q == 0 ? A.b0[c] : T(0), u = q == 0 && !A.zero ? A.u0[c] : T(0);
                V.dg[t] = a[ST_C];
#pragma unroll
                for (int f = 0; f < 6; ++f) V.k[f * V.n + t] = ex[f] ? a[1 + f] : T(0);
                if (q == 0) V.b[t] = b;
                V.u[t] = u;
            }
            if (tid == 0) V.u[V.n] = T(0);
        }
        if (q > 0) {
            const AlignedW W = A.W[q];
            if (tid < 3 * V.nx) V.wx[tid] = W.wx[tid];
            if (tid < 3 * V.ny) V.wy[tid] = W.wy[tid];
            if (tid < 3 * V.nz) V.wz[tid] = W.wz[tid];
        }
    }
    __syncthreads();
    for (int l = 0; l < last; ++l) {
        const SmallView<T> V = small_view(A, mem, l), C = small_view(A, mem, l + 1);
        const TailPlace cells[2] = {small_place(V, tid, 1), small_place(V, tid, 0)};
        small_smooth(A.L[l], V, cells, A.nu1, A.omega[l]);
        // a residual reads only its own right-hand side: it takes its place
        // for the restriction
        T bo[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            bo[p] = T(0);
            const int q = cells[p].q;
            if (q < 0) continue;
            bo[p] = V.b[q];
            V.b[q] = bo[p] - (V.dg[q] * V.u[q] + small_offdiag(V, cells[p]));
        }
        __syncthreads();
        // full weighting onto level l + 1 (as k_restrict_fw_planes; fine
        // values outside the interior carry zero weight)
        for (int t = tid; t < C.n; t += THREADS) {
            int I, J, K;
            small_ijk(C, t, I, J, K);
            double wx[3], wy[3], wz[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                wx[d] = C.wx[3 * I + d];
                wy[d] = C.wy[3 * J + d];
                wz[d] = C.wz[3 * K + d];
            }
            double acc = 0.0;
#pragma unroll
            for (int w = 0; w < 9; ++w) {
                const int j = 2 * J - 1 + w % 3, k = 2 * K - 1 + w / 3;
                const bool in = wy[w % 3] != 0.0 && wz[w / 3] != 0.0;
                const T *row = V.b + (in ? V.nx * (j + V.ny * k) : 0);
                double s = 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const bool ok = in && wx[d] != 0.0;
                    s += wx[d] * (double)(ok ? row[2 * I - 1 + d] : T(0));
                }
                acc += (wz[w / 3] * wy[w % 3]) * s;
            }
            C.b[t] = (T)acc;
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 2; ++p)
            if (cells[p].q >= 0) V.b[cells[p].q] = bo[p];
    }
    // coarsest level: u = A^-1 b (no more rows than lanes)
    {
        const SmallView<T> V = small_view(A, mem, last);
        double s = 0.0;
        if (hb < gb) {
#pragma unroll
            for (int p = 0; p < PRE; ++p) s += inv[p] * (double)V.b[min(hb + p * gb, nb - 1)];
            for (int e0 = hb + PRE * gb; e0 < nb; e0 += 8 * gb) {   // eight loads in flight
                double a[8];
#pragma unroll
                for (int p = 0; p < 8; ++p) a[p] = A.invT[min(e0 + p * gb, nb - 1) * nb + qb];
#pragma unroll
                for (int p = 0; p < 8; ++p) s += e0 + p * gb < nb ? a[p] * (double)V.b[e0 + p * gb] : 0.0;
            }
        }
        part[tid] = s;
        __syncthreads();
        if (tid < nb) {
            s = 0.0;
            for (int p = 0; p < gb; ++p) s += part[p * nb + tid];
            V.u[tid] = (T)s;
        }
        __syncthreads();
    }
    for (int l = last - 1; l >= 0; --l) {
        const SmallView<T> V = small_view(A, mem, l), C = small_view(A, mem, l + 1);
        const TailPlace cells[2] = {small_place(V, tid, 1), small_place(V, tid, 0)};
        const int cy = C.nx, cz = C.nx * C.ny;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (cells[p].q < 0) continue;
            // trilinear prolongation-correction (as k_prolong_tri_planes):
            // 0-based fine cell i takes coarse i / 2 when i is even, else the
            // mean of i / 2 and i / 2 + 1
            int i, j, k;
            small_ijk(V, cells[p].q, i, j, k);
            const T *P0 = C.u + (i / 2 + cy * (j / 2) + cz * (k / 2));
            const int dj = j & 1 ? cy : 0, dk = k & 1 ? cz : 0, di = i & 1;
            auto xy = [&](const T *P) {
                const T a0 = di ? T(0.5) * (P[0] + P[1]) : P[0];
                if (!dj) return a0;
                const T a1 = di ? T(0.5) * (P[dj] + P[dj + 1]) : P[dj];
                return T(0.5) * (a0 + a1);
            };
            const T e0 = xy(P0);
            const T e = dk ? T(0.5) * (e0 + xy(P0 + dk)) : e0;
            V.u[cells[p].q] += e;
        }
        __syncthreads();
        small_smooth(A.L[l], V, cells, A.nu2, A.omega[l]);
    }
    {
        const Lev<T> &L = A.L[0];
        const SmallView<T> V = small_view(A, mem, 0);
        for (int t = tid; t < V.n; t += THREADS) {
            int i, j, k;
            small_ijk(V, t, i, j, k);
            A.u0[(i + 1) + L.sy * (j + 1) + (int)L.sz * (k + 1)] = V.u[t];
        }
    }
}

}  // namespace mps
