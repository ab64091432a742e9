// Coarsest-level solve and Scharfetter-Gummel stencil assembly (gfx950).
#pragma once

#include "mps3d_kernels.h"

namespace mps {

// ------------------------------------------------------------------------
// Bottom solve: performgmres (mgridlib/gmres.f90:197-434) with find_AX and
// gseidel_precond (discretepde.f90:238-337, niter = 1) on the coarsest grid,
// as bottomsolve calls it (mgridsteps.f90:342-355): m = n, one restart,
// classical Gram-Schmidt, Givens rotations, lucky breakdown at 1e-25.
//
// One workgroup runs the whole solve. Vector updates are spread over the
// workgroup; every inner product is summed by one lane in the reference's
// memory order (its products formed in parallel), so the coarse solve
// reproduces the reference's rounding. The kd Gram-Schmidt products of
// Arnoldi step kd all take the unmodified w (classical Gram-Schmidt), so
// they run at once, one lane each, against w held in LDS. The coarsest grid
// holds at most kBottomMax cells.
// ------------------------------------------------------------------------
constexpr int kBottomMax = 512;
// Krylov dimensions up to this keep the Hessenberg matrix and the Givens
// arrays in LDS (the reference's coarse solves use m = n, which is 8-64 on
// the usual process grids); larger m keep them in the work buffer
constexpr int kBottomLdsM = 64;
// Coarse grids of up to this many cells with m <= kBottomLdsM also keep an
// interior-only copy of the Krylov basis in LDS (column stride n + 1), so
// the Gram-Schmidt products and the orthogonalised vector read no global
// memory; the ghosted basis stays in the work buffer for the operator.
constexpr int kBottomLdsN = 64;

template <typename T>
__host__ __device__ inline long long bottom_work_elems(int m, long long ng)
{
    return (long long)(m + 1) * ng + 8 * ng + (long long)(m + 1) * m + 4LL * (m + 1);
}

// performgmres with nrestarts restarts of GMRES(m); the coarse solve uses
// m = n, nrestarts = 1 and tol = ERRTOLR*0.0001 (mgridsteps.f90:305, :342-343).
// LM: m <= kBottomLdsM, the Hessenberg and Givens arrays in LDS. A compile-
// time choice, so they are addressed as LDS (a pointer chosen at run time
// between LDS and global memory is a generic one, and every access through it
// a flat instruction).
template <typename T, int OP, bool VEL, bool REAC, bool LM>
__global__ void __launch_bounds__(kBlock) k_bottom(Lev<T> L, T *u, const T *__restrict__ b, T *work, int m,
                                                  int nrestarts, T tol, int *status)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int n = nx * ny * nz;
    const long long ng = (long long)(nx + 2) * (ny + 2) * (nz + 2);
    T *V = work;
    T *x = V + (long long)(m + 1) * ng;
    T *x0 = x + ng;
    T *r0 = x0 + ng;
    T *r = r0 + ng;
    T *av = r + ng;
    T *w = av + ng;
    T *wj = w + ng;
    T *mb = wj + ng;
    __shared__ T sH[(kBottomLdsM + 1) * kBottomLdsM];
    __shared__ T sg[4 * (kBottomLdsM + 1)];
    const bool lds = LM;
    T *H = LM ? sH : mb + ng;
    T *cs = LM ? sg : H + (long long)(m + 1) * m;
    T *sn = cs + (m + 1);
    T *be = sn + (m + 1);
    T *y = be + (m + 1);
    __shared__ T sh[2];
    __shared__ int cmap[kBottomMax];   // interior cell q (i fastest) -> ghosted index
    __shared__ T pr[kBottomMax];       // products of one inner product
    __shared__ T wsh[kBottomMax];      // w of the current Arnoldi step, by cell
    __shared__ T sV[(kBottomLdsM + 1) * (kBottomLdsN + 1)];
    const bool vlds = lds && n <= kBottomLdsN;
    const int ldv = n + 1;
    const int tid = threadIdx.x, nt = blockDim.x;

    auto cidx = [&](int q, int &i, int &j, int &k) {
        i = q % nx + 1;
        j = (q / nx) % ny + 1;
        k = q / (nx * ny) + 1;
        return (long long)i + (long long)L.sy * j + L.sz * k;
    };
    auto zero = [&](T *v) {
        for (long long q = tid; q < ng; q += nt) v[q] = T(0);
        __syncthreads();
    };
    auto apply = [&](T *out, const T *in) {  // out interior = A in
        for (int q = tid; q < n; q += nt) {
            int i, j, k;
            long long c = cidx(q, i, j, k);
            T dg, of;
            row<T, OP, VEL, REAC>(L, in, i, j, k, c, dg, of);
            out[c] = dg * in[c] + of;
        }
        __syncthreads();
    };
    // gseidel_precond, niter = 1 (discretepde.f90:238-337), from out = 0:
    // the interior of out is cleared, then the red cells take
    // (in - of) / dg with of formed from the cleared black neighbours (as in
    // the reference: a non-finite coefficient makes it NaN there too), then
    // the black cells from the new red ones. Invariant: every buffer that
    // precond writes (mb, r, w) has zero ghost entries, set once at the
    // kernel's start and never written afterwards; explicit (OP_STENCIL)
    // rows of boundary cells multiply those ghosts by their zero
    // coefficients.
    auto precond = [&](T *out, const T *in) {
        if (n == 1) {
            if (tid == 0) {
                int i, j, k;
                long long c = cidx(0, i, j, k);
                T dg, of;
                row<T, OP, VEL, REAC>(L, in, i, j, k, c, dg, of);
                out[c] = in[c] / dg;
            }
            __syncthreads();
            return;
        }
        for (int q = tid; q < n; q += nt) out[cmap[q]] = T(0);
        __syncthreads();
        for (int q = tid; q < n; q += nt) {   // red cells from the cleared black ones
            int i, j, k;
            long long c = cidx(q, i, j, k);
            if (((i + j + k) & 1) != 1) continue;
            T dg, of;
            row<T, OP, VEL, REAC>(L, out, i, j, k, c, dg, of);
            out[c] = (in[c] - of) / dg;
        }
        __syncthreads();
        for (int q = tid; q < n; q += nt) {   // black cells from the new red ones
            int i, j, k;
            long long c = cidx(q, i, j, k);
            if (((i + j + k) & 1) != 0) continue;
            T dg, of;
            row<T, OP, VEL, REAC>(L, out, i, j, k, c, dg, of);
            out[c] = (in[c] - of) / dg;
        }
        __syncthreads();
    };
    for (int q = tid; q < n; q += nt) {
        int i, j, k;
        cmap[q] = (int)cidx(q, i, j, k);
    }
    __syncthreads();
    auto dot = [&](const T *a, const T *c2) {  // products in parallel, one lane sums in order
        for (int q = tid; q < n; q += nt) pr[q] = a[cmap[q]] * c2[cmap[q]];
        __syncthreads();
        if (tid == 0) {
            T s = T(0);
#pragma unroll 8
            for (int q = 0; q < n; ++q) s = s + pr[q];
            sh[0] = s;
        }
        __syncthreads();
        T s = sh[0];
        __syncthreads();
        return s;
    };
#define HM(i_, j_) H[(long long)((i_) - 1) + (long long)(m + 1) * ((j_) - 1)]

    if (tid == 0) *status = 0;
    zero(x);
    zero(r0);
    zero(av);   // apply and precond write interiors only: the ghost entries
    zero(w);    // of these stay zero for the whole solve
    zero(r);
    zero(mb);
    for (int q = tid; q < n; q += nt) {
        int i, j, k;
        long long c = cidx(q, i, j, k);
        x[c] = u[c];
        r0[c] = b[c];
    }
    __syncthreads();
    for (int rs = 1; rs <= nrestarts; ++rs) {
        for (long long q = tid; q < (long long)(m + 1) * ng; q += nt) V[q] = T(0);
        for (long long q = tid; q < (long long)(m + 1) * m; q += nt) H[q] = T(0);
        for (int q = tid; q < m + 1; q += nt) {
            cs[q] = T(0);
            sn[q] = T(0);
            be[q] = T(0);
            y[q] = T(0);
        }
        __syncthreads();
        // Minvb from b with zero ghosts (r0 is reused as the ghosted b)
        zero(r0);
        for (int q = tid; q < n; q += nt) {
            int i, j, k;
            long long c = cidx(q, i, j, k);
            r0[c] = b[c];
        }
        __syncthreads();
        precond(mb, r0);
        const T bnorm = sqrt(dot(mb, mb));
        if (bnorm == T(0)) {
            zero(x);
            break;
        }
        for (long long q = tid; q < ng; q += nt) x0[q] = x[q];
        __syncthreads();
        apply(av, x0);
        zero(r0);
        for (int q = tid; q < n; q += nt) {
            int i, j, k;
            long long c = cidx(q, i, j, k);
            r0[c] = b[c] - av[c];
        }
        __syncthreads();
        precond(r, r0);
        const T beta = sqrt(dot(r, r));
        if (tid == 0) be[0] = beta;
        __syncthreads();
        if (fabs((double)beta) < (double)tol) break;
        for (long long q = tid; q < ng; q += nt) V[q] = r[q] / beta;
        if (vlds)
            for (int q = tid; q < n; q += nt) sV[q] = r[cmap[q]] / beta;
        __syncthreads();
        int optk = m;
        int lucky = 0;
        T residnorm = T(0);
        for (int kd = 1; kd <= m; ++kd) {
            const T *vj = V + ng * (long long)(kd - 1);
            apply(av, vj);
            precond(w, av);
            // The serial loops below are unrolled so that their loads issue
            // ahead of the dependent chain; the summation order is unchanged.
            // classical Gram-Schmidt: h_ii = <w, v_ii> for ii = 1..kd, one
            // lane each, then wj = w - h_1 v_1 - h_2 v_2 - ... in that order
            for (int q = tid; q < n; q += nt) wsh[q] = w[cmap[q]];
            __syncthreads();
            for (int ii = 1 + tid; ii <= kd; ii += nt) {
                T h = T(0);
                if (vlds) {
                    const T *vi = sV + ldv * (ii - 1);
#pragma unroll 8
                    for (int q = 0; q < n; ++q) h = h + wsh[q] * vi[q];
                } else {
                    const T *vi = V + ng * (long long)(ii - 1);
#pragma unroll 8
                    for (int q = 0; q < n; ++q) h = h + wsh[q] * vi[cmap[q]];
                }
                HM(ii, kd) = h;
            }
            __syncthreads();
            T hn;
            if (vlds) {
                // wj by cell over the interior (the ghost entries of every
                // basis vector are zero), kept in wsh, with the products of
                // <wj, wj> formed beside it and summed in order by one lane
                for (int q = tid; q < n; q += nt) {
                    T t = wsh[q];
#pragma unroll 8
                    for (int ii = 1; ii <= kd; ++ii) t = t - HM(ii, kd) * sV[ldv * (ii - 1) + q];
                    wsh[q] = t;
                    pr[q] = t * t;
                }
                __syncthreads();
                if (tid == 0) {
                    T s2 = T(0);
#pragma unroll 8
                    for (int q = 0; q < n; ++q) s2 = s2 + pr[q];
                    sh[0] = s2;
                }
                __syncthreads();
                hn = sqrt(sh[0]);
            } else {
                for (long long q = tid; q < ng; q += nt) {
                    T t = w[q];
                    for (int ii = 1; ii <= kd; ++ii) t = t - HM(ii, kd) * V[ng * (long long)(ii - 1) + q];
                    wj[q] = t;
                }
                __syncthreads();
                hn = sqrt(dot(wj, wj));
            }
            int nanflag = 0;
            if (hn > T(1e-25)) {
                T *vn = V + ng * (long long)kd;
                if (vlds) {
                    for (int q = tid; q < n; q += nt) {
                        const T v = wsh[q] / hn;
                        vn[cmap[q]] = v;
                        sV[ldv * kd + q] = v;
                    }
                } else {
                    for (long long q = tid; q < ng; q += nt) vn[q] = wj[q] / hn;
                }
            } else if (!(hn != hn) && !((hn / hn != T(1)) && hn != T(0))) {
                lucky = 1;
            } else {
                nanflag = 1;
            }
            __syncthreads();
            if (nanflag) {
                if (tid == 0) *status = -1;
                return;
            }
            if (tid == 0) {  // triangularize (gmres.f90:159-195)
                HM(kd + 1, kd) = hn;
                // the rotated entry ii+1 becomes the next step's entry ii:
                // carried in a register, the chain touches memory only to
                // load the untouched entries and store the finished ones
                T hc = HM(1, kd);
#pragma unroll 8
                for (int ii = 1; ii <= kd - 1; ++ii) {
                    const T hn1 = HM(ii + 1, kd), c = cs[ii - 1], s = sn[ii - 1];
                    const T t = c * hc + s * hn1;
                    hc = -s * hc + c * hn1;
                    HM(ii, kd) = t;
                }
                if (kd > 1) HM(kd, kd) = hc;
                T rr = HM(kd, kd), ss = HM(kd + 1, kd), c, s;
                if (rr == T(0)) {
                    c = T(0);
                    s = T(1);
                } else {
                    c = rr / sqrt(rr * rr + ss * ss);
                    s = ss / sqrt(rr * rr + ss * ss);
                }
                HM(kd, kd) = c * HM(kd, kd) + s * HM(kd + 1, kd);
                HM(kd + 1, kd) = T(0);
                cs[kd - 1] = c;
                sn[kd - 1] = s;
                be[kd] = -s * be[kd - 1];
                be[kd - 1] = c * be[kd - 1];
                sh[1] = fabs(be[kd]);
            }
            __syncthreads();
            residnorm = sh[1];
            __syncthreads();
            if (lucky) {
                optk = kd;
                break;
            }
        }
        if (tid == 0) {  // uppertrisolve (gmres.f90:124-142)
            for (int ii = optk; ii >= 1; --ii) {
                y[ii - 1] = be[ii - 1];
                for (int jj = ii + 1; jj <= optk; ++jj) y[ii - 1] = y[ii - 1] - HM(ii, jj) * y[jj - 1];
                y[ii - 1] = y[ii - 1] / HM(ii, ii);
            }
        }
        __syncthreads();
        for (long long q = tid; q < ng; q += nt) {
            T xv = x0[q];
            for (int jj = 1; jj <= optk; ++jj) xv = xv + y[jj - 1] * V[ng * (long long)(jj - 1) + q];
            x[q] = xv;
        }
        __syncthreads();
        if (residnorm / bnorm <= tol || lucky) break;
    }
    for (int q = tid; q < n; q += nt) {
        int i, j, k;
        long long c = cidx(q, i, j, k);
        u[c] = x[c];
    }
#undef HM
}

// ------------------------------------------------------------------------
// The same solve for at most kWaveN cells and m <= kWaveN in one wavefront,
// bit for bit k_bottom's result. Lane q owns cell q; the level's row of that
// cell (diagonal, face conductances, face velocities) stays in registers
// for the whole solve, the Krylov basis, the Hessenberg matrix and the
// vectors that other lanes read stay in LDS, and nothing waits on global
// memory or on a workgroup barrier between the first load and the last
// store. What bounds it is the instruction count of one wave (4 cycles each)
// on the reference's serial summation order: an Arnoldi step is two chains
// of n dependent additions (the kd Gram-Schmidt products, one per lane, and
// the norm) and one of kd subtractions. Those loops are laid out flat in
// chunks that a uniform branch skips, with the next chunk's LDS loads ahead
// of the additions. Two things that the reference does step by step on
// one value at a time are done once, in another loop order with the same
// operands and results: the Givens rotations of all columns after the last
// Arnoldi step (the iteration reads none of them), one column per lane, and
// the products of the back substitution's rows.
// Sums run over whole chunks: the entries past n (or past kd) are zero, and
// adding or subtracting +0 leaves every partial sum as it is (a sum that
// starts at +0 is never -0). 64 cells, 64 steps: 148 us, of it 110 us in the
// Arnoldi steps (4200 cycles each: products 1230, subtractions 1020, norm
// 840, operator and preconditioner 830), rotations 15 us, back substitution
// 22 us; with rolled loops and broadcasts through ds_bpermute 204 us.
// ------------------------------------------------------------------------
constexpr int kWaveN = 64;            // one cell per lane
constexpr int kWaveLd = kWaveN + 2;   // entries kWaveN, kWaveN + 1 of a row stay zero

template <typename T>
struct alignas(2 * sizeof(T)) PairT {
    T a, b;
};

// LDS operations of one wave complete in order: between a lane's write and
// another lane's read only the compiler has to be held
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the value of lane q (uniform)
__device__ __forceinline__ double lane_value(double v, int q)
{
    const long long b = __builtin_bit_cast(long long, v);
    const unsigned lo = __builtin_amdgcn_readlane((int)b, q), hi = __builtin_amdgcn_readlane((int)(b >> 32), q);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float lane_value(float v, int q)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), q));
}

// s + a[0] c[0] + a[1] c[1] + ... (FORM 1), s + a[0] + a[1] + ... (FORM 0) or
// s - a[0] - a[1] - ... (FORM -1), n terms in order, in chunks of 16 (a, c
// aligned to a pair, zero past n up to the next chunk)
template <typename T, int FORM>
__device__ __forceinline__ T serial_sum(T s, const T *a, const T *c, int n)
{
    constexpr int K = 8, NC = kWaveN / (2 * K);
    const PairT<T> *pa = reinterpret_cast<const PairT<T> *>(a);
    const PairT<T> *pc = reinterpret_cast<const PairT<T> *>(c);
    PairT<T> ra[NC][K], rc[NC][K];
    auto load = [&](int g) {
#pragma unroll
        for (int t = 0; t < K; ++t) {
            ra[g][t] = pa[g * K + t];
            if (FORM == 1) rc[g][t] = pc[g * K + t];
        }
    };
    auto add = [&](int g) {
#pragma unroll
        for (int t = 0; t < K; ++t) {
            if (FORM == -1) {
                s = s - ra[g][t].a;
                s = s - ra[g][t].b;
            } else {
                s = s + (FORM == 1 ? ra[g][t].a * rc[g][t].a : ra[g][t].a);
                s = s + (FORM == 1 ? ra[g][t].b * rc[g][t].b : ra[g][t].b);
            }
        }
    };
    load(0);
    if (n > 16) {
        load(1);
        add(0);
        if (n > 32) {
            load(2);
            add(1);
            if (n > 48) {
                load(3);
                add(2);
                add(3);
            } else {
                add(2);
            }
        } else {
            add(1);
        }
    } else {
        add(0);
    }
    return s;
}

// t - h[0] V[0][lane] - h[1] V[1][lane] - ... in that order, kd terms in
// chunks of 8 (h zero past kd, V finite)
template <typename T, int G = 0>
__device__ __forceinline__ T serial_axpy(T t, const T *h, const T (*V)[kWaveLd], int lane, int kd, const PairT<T> *h0,
                                         const T *v0)
{
    constexpr int K = 8;
    PairT<T> h1[K / 2];
    T v1[K];
    if constexpr (8 * (G + 1) < kWaveN) {
        const PairT<T> *ph = reinterpret_cast<const PairT<T> *>(h) + K / 2 * (G + 1);
#pragma unroll
        for (int p = 0; p < K / 2; ++p) h1[p] = ph[p];
#pragma unroll
        for (int p = 0; p < K; ++p) v1[p] = V[K * (G + 1) + p][lane];
    }
#pragma unroll
    for (int p = 0; p < K / 2; ++p) {
        t = t - h0[p].a * v0[2 * p];
        t = t - h0[p].b * v0[2 * p + 1];
    }
    if constexpr (8 * (G + 1) < kWaveN) {
        if (kd > 8 * (G + 1)) return serial_axpy<T, G + 1>(t, h, V, lane, kd, h1, v1);
    }
    return t;
}

template <typename T, int OP, bool VEL, bool REAC>
__global__ void __launch_bounds__(kWaveN) k_bottom_wave(Lev<T> L, T *u, const T *__restrict__ b, int m, int nrestarts,
                                                       T tol, int *status)
{
    // basis vectors by row, Hessenberg columns by row (entry ii of column kd
    // at sH[kd][ii], 0-based)
    __shared__ alignas(16) T sV[kWaveN + 1][kWaveLd];
    __shared__ alignas(16) T sH[kWaveN][kWaveLd];
    __shared__ alignas(16) T sr[kWaveLd];   // red values of the preconditioner
    __shared__ alignas(16) T sw[kWaveLd];   // the vector or products that every lane reads
    const int lane = threadIdx.x;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int n = nx * ny * nz;
    const bool own = lane < n;
    const int q0 = own ? lane : 0;
    const int i = q0 % nx + 1, j = (q0 / nx) % ny + 1, k = q0 / (nx * ny) + 1;
    const long long c = (long long)i + (long long)L.sy * j + L.sz * k;
    const bool red = ((i + j + k) & 1) == 1;
    // the six neighbours in a row of sV, sr: kWaveN (a zero) where the face
    // does not exist
    const bool ex[6] = {i > 1, i < nx, j > 1, j < ny, k > 1, k < nz};
    const int nb[6] = {ex[0] ? lane - 1 : kWaveN,       ex[1] ? lane + 1 : kWaveN,  ex[2] ? lane - nx : kWaveN,
                       ex[3] ? lane + nx : kWaveN,      ex[4] ? lane - nx * ny : kWaveN,
                       ex[5] ? lane + nx * ny : kWaveN};
    // The row. face_right and face_left add 0 - u kq ab and, on the upwind
    // side, -+ vh u ab per face (kq = kh / d): a face's two multipliers of
    // u carry those signs, and a term that does not exist has multiplier 0
    // (its +-0 leaves the sum as it is). Explicit rows: kq = st.
    T dg, kq[6], vq[6], ab[3];
    const T bc = own ? b[c] : T(0);
    T x = own ? u[c] : T(0);
    {
        // (every load first: the ghosted arrays hold every neighbour, so no
        // load waits on a test of the face before it)
        const long long st[3] = {1, L.sy, L.sz};
        const T *v3[3] = {L.vx, L.vy, L.vz};
        const T h[3] = {L.dx, L.dy, L.dz};
        const T a0[3] = {L.ax, L.ay, L.az}, a1[3] = {L.axb, L.ayb, L.azb}, i0[3] = {L.ix0, L.iy0, L.iz0};
        T Dn[6], vn[6], vc[3], Dc = T(0), rc = T(0);
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const long long o = (f & 1) ? c + st[f / 2] : c - st[f / 2];
            if (OP == OP_STENCIL) kq[f] = L.st[1 + f][c];
            else Dn[f] = L.D[o];
            if (VEL) vn[f] = v3[f / 2][o];
            if (VEL && !(f & 1)) vc[f / 2] = v3[f / 2][c];
        }
        if (OP == OP_STENCIL) dg = L.st[ST_C][c];
        else Dc = L.D[c];
        if (OP != OP_STENCIL && REAC) rc = L.reac[c];
        if (OP != OP_STENCIL) {
            // the diagonal in row()'s order: per direction the two faces,
            // then the wall terms; reaction and time last
            T d = T(0);
#pragma unroll
            for (int f = 0; f < 6; ++f) {
                const int q = f / 2;
                const bool edge = !ex[2 * q] || !ex[2 * q + 1];
                ab[q] = (OP == OP_ALIGNED && edge) ? a1[q] : a0[q];
                // (left + right, in that order, as the face functions add)
                const T kf = (T(0.5) * ((f & 1) ? Dc + Dn[f] : Dn[f] + Dc)) / h[q];
                T t = T(0) + kf * ab[q];
                kq[f] = ex[f] ? -kf : T(0);
                if (VEL) {
                    const T vh = T(0.5) * ((f & 1) ? vc[q] + vn[f] : vn[f] + vc[q]);
                    const bool pos = vh > T(0);
                    // the upwind cell of the face is the left one where vh > 0
                    if (f & 1) t = pos ? t + vh * ab[q] : t;
                    else t = pos ? t : t - vh * ab[q];
                    vq[f] = (ex[f] && pos == !(f & 1)) ? ((f & 1) ? vh : -vh) : T(0);
                }
                if (ex[f]) d = d + t;
                if (f & 1) {
                    if (!ex[f - 1])
                        bc_row<T, OP, VEL>(L.bc[f - 1], false, Dc, VEL ? vc[q] : T(0), h[q], ab[q], i0[q], d);
                    if (!ex[f]) bc_row<T, OP, VEL>(L.bc[f], true, Dc, VEL ? vc[q] : T(0), h[q], ab[q], i0[q], d);
                }
            }
            if (REAC) d = d - rc;
            if (L.timederiv) d = d + T(1) / L.dt;
            dg = d;
        }
    }
    // off-diagonal sum of this lane's row over neighbour values in a row of LDS
    auto offdiag = [&](const T *p) {
        T un[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) un[f] = p[nb[f]];
        T o = T(0);
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            if (OP == OP_STENCIL) {
                o = o + kq[f] * un[f];
            } else {
                T t = un[f] * kq[f] * ab[f / 2];
                if (VEL) t = t + vq[f] * un[f] * ab[f / 2];
                o = o + t;
            }
        }
        return o;
    };
    sr[lane] = T(0);
    for (int q = 0; q <= kWaveN; ++q) sV[q][lane] = T(0);
    sV[lane][kWaveN] = sV[lane][kWaveN + 1] = T(0);
    if (lane < 2) sr[kWaveN + lane] = T(0), sw[kWaveN + lane] = T(0);
    wave_fence();
    const T of0 = offdiag(sr);   // of a red cell: its black neighbours are cleared
    // gseidel_precond of the vector whose entry of this cell is `in`
    auto precond = [&](T in) {
        T v = (in - of0) / dg;
        sr[lane] = (own && red) ? v : T(0);
        wave_fence();
        const T o = offdiag(sr);
        if (!red) v = (in - o) / dg;
        wave_fence();
        return own ? v : T(0);
    };
    auto norm = [&](T v) {
        sw[lane] = v * v;
        wave_fence();
        const T s = serial_sum<T, 0>(T(0), sw, sw, n);
        wave_fence();
        return sqrt(s);
    };

    if (lane == 0) *status = 0;
    for (int rs = 1; rs <= nrestarts; ++rs) {
        const T bnorm = norm(precond(bc));
        if (bnorm == T(0)) {
            x = T(0);
            break;
        }
        const T x0 = x;
        sw[lane] = x0;
        wave_fence();
        const T av0 = dg * x0 + offdiag(sw);
        wave_fence();
        const T r = precond(own ? bc - av0 : T(0));
        const T beta = norm(r);
        if (fabs((double)beta) < (double)tol) break;
        T v = own ? r / beta : T(0);   // the newest basis vector's entry
        sV[0][lane] = v;
        wave_fence();
        int optk = m, lucky = 0;
        for (int kd = 1; kd <= m; ++kd) {
            const T av = dg * v + offdiag(sV[kd - 1]);
            const T w = precond(own ? av : T(0));
            sw[lane] = w;
            wave_fence();
            // h_ii = <w, v_ii>, lane ii - 1 (of the rows filled so far)
            T *hk = sH[kd - 1];
            const T h = serial_sum<T, 1>(T(0), sw, sV[lane], n);
            hk[lane] = lane < kd ? h : T(0);
            wave_fence();
            // w - h_1 v_1 - h_2 v_2 - ... in that order
            PairT<T> h0[4];
            T v0[8];
#pragma unroll
            for (int p = 0; p < 8; ++p) v0[p] = sV[p][lane];
#pragma unroll
            for (int p = 0; p < 4; ++p) h0[p] = reinterpret_cast<const PairT<T> *>(hk)[p];
            const T t = serial_axpy<T>(w, hk, sV, lane, kd, h0, v0);
            const T hn = norm(t);
            if (hn > T(1e-25)) {
                v = own ? t / hn : T(0);
                sV[kd][lane] = v;
            } else if (!(hn != hn) && !((hn / hn != T(1)) && hn != T(0))) {
                lucky = 1;
            } else {
                if (lane == 0) *status = -1;
                return;
            }
            if (lane == 0) hk[kd] = hn;
            wave_fence();
            if (lucky) {
                optk = kd;
                break;
            }
        }
        // triangularize (gmres.f90:159-195): rotation ii is formed from
        // column ii and applied to the columns after it, lane = column; hc is
        // the column's entry of row ii after the rotations before
        T bl = T(0), bcur = beta;   // be(ii) of lane ii, be(ii + 1) so far
        T rdiag = T(1), rsup = T(0);   // R(lane, lane), R(lane - 1, lane)
        {
            T *const col = sH[min(lane, optk - 1)];
            T hc = col[0], hn1 = col[1];
            for (int ii = 0; ii < optk; ++ii) {
                const T hn2 = col[min(ii + 2, kWaveN)];
                const T rr = lane_value(hc, ii), ss = lane_value(hn1, ii);
                T cs, sn;
                if (rr == T(0)) {
                    cs = T(0);
                    sn = T(1);
                } else {
                    const T den = sqrt(rr * rr + ss * ss);
                    cs = rr / den;
                    sn = ss / den;
                }
                const T t = cs * hc + sn * hn1;
                hc = -sn * hc + cs * hn1;
                hn1 = hn2;
                if (lane == ii) {
                    rdiag = t;
                    bl = cs * bcur;
                }
                if (lane == ii + 1) rsup = t;
                if (lane > ii && lane < optk) col[ii] = t;
                bcur = -sn * bcur;
            }
        }
        const T residnorm = fabs(bcur);
        wave_fence();
        // uppertrisolve (gmres.f90:124-142): row ii subtracts its products
        // in ascending columns. Those of the columns past ii + 1 are formed
        // (lane = column) and stored a row ahead, so that only y(ii + 1)'s
        // own is formed when it is known; the sum runs over whole chunks of
        // 16 (zeros before column ii + 2 and past optk)
        T y = T(0), yi = T(0);
        sw[lane] = T(0);
        T hrow = sH[lane][max(optk - 2, 0)];   // R(ii - 1, lane) at row ii
        wave_fence();
        for (int ii = optk - 1; ii >= 0; --ii) {
            T s = lane_value(bl, ii);
            if (ii + 1 < optk) {
                s = s - lane_value(rsup, ii + 1) * yi;
                const int j0 = (ii + 2) & ~15;
                if (j0 < optk) s = serial_sum<T, -1>(s, sw + j0, sw, optk - j0);
            }
            wave_fence();
            sw[lane] = (lane > ii && lane < optk) ? hrow * y : T(0);
            hrow = sH[lane][max(ii - 2, 0)];
            yi = s / lane_value(rdiag, ii);
            if (lane == ii) y = yi;
            wave_fence();
        }
        sw[lane] = y;
        wave_fence();
        T xv = x0;
#pragma unroll 8
        for (int jj = 0; jj < optk; ++jj) xv = xv + sw[jj] * sV[jj][lane];
        x = xv;
        wave_fence();
        if (residnorm / bnorm <= tol || lucky) break;
    }
    if (own) u[c] = x;
}

// ------------------------------------------------------------------------
// Scharfetter-Gummel operator rows
// ------------------------------------------------------------------------

// Bernoulli function B(x) = x/(e^x - 1), evaluated in FP64 with expm1 and a
// Taylor series near 0 (B = 1 - x/2 + x^2/12 - x^4/720 + ...) so that the
// small-drift limit stays exact.
__device__ __forceinline__ double bernoulli(double x)
{
    const double ax = fabs(x);
    if (ax < 1e-3) {
        const double x2 = x * x;
        return 1.0 - 0.5 * x + x2 * (1.0 / 12.0 - x2 * (1.0 / 720.0));
    }
    if (x > 700.0) return x * exp(-x);
    return x / expm1(x);
}

// SG weights of one face (wL multiplies the left value, wR the right) in
// the form of find_sg_exponential_flux (mps1d/source/convdiff.f90:10-64):
// c = mean velocity, D = harmonic mean with the reference's 1e-10 guard,
// pure upwind for vanishing D, central diffusion for vanishing Peclet.
__device__ __forceinline__ void sg_weights(double cL, double cR, double DL, double DR, double d, double &wL,
                                           double &wR)
{
    const double eps = 1e-10;
    const double ch = 0.5 * (cL + cR);
    const double Dh = 2.0 * DL * DR / (DL + DR + eps);
    if (fabs(Dh) < eps) {
        const double sgn = ch <= 0.0 ? -1.0 : 1.0;
        wL = cL * 0.5 * (1.0 + sgn);
        wR = cR * 0.5 * (1.0 - sgn);
        return;
    }
    const double Pe = ch * d / Dh;
    const double g = Dh / d;
    if (fabs(Pe) < eps) {
        wL = g;
        wR = -g;
        return;
    }
    wL = g * bernoulli(-Pe);
    wR = -g * bernoulli(Pe);
}

// Assembles the 7-point SG rows of one level: each interior face carries
// the flux F = wL u_L + wR u_R (positive along +axis); row L gains F/w_L,
// row R loses F/w_R. Physical faces keep the reference's boundary rows
// (DIRC diffusion to the wall plus upwind outflow, ZGRD outflow). Reaction
// and 1/dt sit on the diagonal. transpose != 0 stores A^T. The FP32 cycle's
// copy of the rows (st32, nullable) is written in the same pass. Only
// interior entries are written: the arrays are zero from their allocation on.
struct RowArrays {
    double *st[ST_N];
    float *st32[ST_N];
};

template <int OP>
__global__ void __launch_bounds__(kBlock) k_sg_stencil(Lev<double> L, RowArrays S, int transpose)
{
    int i, j, k;
    long long c;
    if (!cell_of(L, i, j, k, c)) return;
    double *const *st = S.st;
    double a[ST_N];
    for (int q = 0; q < ST_N; ++q) a[q] = 0.0;
    double d = 0.0;
    const double *D = L.D;
    const double Dc = D[c];
    const double *vel[3] = {L.vx, L.vy, L.vz};
    const long long s[3] = {1, L.sy, L.sz};
    const int idx[3] = {i, j, k};
    const int nn[3] = {L.nx, L.ny, L.nz};
    const double h[3] = {L.dx, L.dy, L.dz};
    const double ai[3] = {L.ax, L.ay, L.az};
    const double ab[3] = {L.axb, L.ayb, L.azb};
    const double i0[3] = {L.ix0, L.iy0, L.iz0};
    for (int dim = 0; dim < 3; ++dim) {
        const bool edge = idx[dim] == 1 || idx[dim] == nn[dim];
        const double abv = (OP == OP_ALIGNED && edge) ? ab[dim] : ai[dim];
        const double vc = vel[dim] ? vel[dim][c] : 0.0;
        if (idx[dim] > 1) {  // face (c-s | c): this cell is R
            const long long m = c - s[dim];
            double wL, wR;
            sg_weights(vel[dim] ? vel[dim][m] : 0.0, vc, D[m], Dc, h[dim], wL, wR);
            d = d - wR * abv;
            a[1 + 2 * dim] = -wL * abv;
        }
        if (idx[dim] < nn[dim]) {  // face (c | c+s): this cell is L
            const long long p = c + s[dim];
            double wL, wR;
            sg_weights(vc, vel[dim] ? vel[dim][p] : 0.0, Dc, D[p], h[dim], wL, wR);
            d = d + wL * abv;
            a[2 + 2 * dim] = wR * abv;
        }
        if (idx[dim] == 1) bc_row<double, OP, true>(L.bc[2 * dim], false, Dc, vc, h[dim], abv, i0[dim], d);
        if (idx[dim] == nn[dim]) bc_row<double, OP, true>(L.bc[2 * dim + 1], true, Dc, vc, h[dim], abv, i0[dim], d);
    }
    if (L.reac) d = d - L.reac[c];
    if (L.timederiv) d = d + 1.0 / L.dt;
    a[ST_C] = d;
    if (!transpose) {
#pragma unroll
        for (int q = 0; q < ST_N; ++q) {
            st[q][c] = a[q];
            if (S.st32[q]) S.st32[q][c] = (float)a[q];
        }
        return;
    }
    st[ST_C][c] = a[ST_C];
    if (i > 1) st[ST_XP][c - 1] = a[ST_XM];
    if (i < L.nx) st[ST_XM][c + 1] = a[ST_XP];
    if (j > 1) st[ST_YP][c - L.sy] = a[ST_YM];
    if (j < L.ny) st[ST_YM][c + L.sy] = a[ST_YP];
    if (k > 1) st[ST_ZP][c - L.sz] = a[ST_ZM];
    if (k < L.nz) st[ST_ZM][c + L.sz] = a[ST_ZP];
}

// ------------------------------------------------------------------------
// Dense inverse of the coarsest operator on the device: the coarse solve of
// a V-cycle is then one small matrix-vector product (k_bottom_dense). On
// the reference hierarchy in fast arithmetic it stands for the reference's
// coarse GMRES (m = n, one restart, tol 1e-15, mgridsteps.f90:342-355), which
// is an exact solve up to rounding.
//
// One workgroup assembles A from the level's 7-point rows and inverts it in
// place by Gauss-Jordan elimination with partial pivoting. For n <= kInvRegsN
// the whole matrix lives in the workgroup's registers (512 KB per CU; its
// LDS would hold 141 rows): lane (tr, tc) of a 16 x 32 grid owns the entries
// (tr + 16 a, tc + 32 b), a < 2 E, b < E, and a pivot step passes one column
// and one row through LDS (two buffers, two barriers). Every wave finds the
// pivot by itself, a maximum over keys (|value| with its low 8 bits replaced
// by 255 - row, so near-ties go to the lowest row) in cross-lane moves of
// the vector unit. Rows stay where they are; which row took step kk is
// recorded and undone in the final scatter, which moves the same values as
// swapping rows and swapping columns back. A pivot below kPivotFloor of its
// column's largest entry (or a NaN) sets *status = -1: whether such an
// operator is singular depends on how its elimination rounds, and the caller
// leaves the answer, and the inverse, to host_bottom_inverse.
// 27 cells 21 us, 64 cells 52 us (98 us with the matrix in LDS, one column
// per lane), 128 cells 162 us, 210 cells 444 us (2.1 us per pivot; 1024 lanes
// with 49 entries each spill: 1000 us). On the host, with the rows copied
// there and the inverse back, the 210-cell one held a 6.6 ms species step up
// for more than 2 ms.
// ------------------------------------------------------------------------
constexpr int kInvRegsN = 224;
constexpr int kInvThreads = 512;
// An elimination with partial pivoting ends in an exact zero only where it
// leaves rounding errors of the column, some n eps of its largest entry: no-
// flux operators of 2 to 224 cells end at 5e-14 of it at most, in this
// kernel's fused arithmetic too; one plane of DIRC faces keeps them above 0.05.
constexpr double kPivotFloor = 1.0 / (1 << 30);
constexpr int kDenseThreads = 1024;

// max over the wave of a key >= 0, in lane 63 (row shifts within 16 lanes,
// then row broadcasts; lanes without a source take 0)
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_max(unsigned long long v)
{
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false);
    const unsigned long long o = ((unsigned long long)hi << 32) | lo;
    return o > v ? o : v;
}

template <int E>
__global__ void __launch_bounds__(kInvThreads) k_dense_inverse_regs(Lev<double> L, RowArrays S, double *Ainv,
                                                                    double *AinvT, int *status)
{
    constexpr int N = 32 * E, A = 2 * E, B = E;
    __shared__ double scol[2][N], srow[2][N];
    __shared__ double floor_of[N];   // the least pivot of a column that counts as one
    __shared__ int perm[N], pos[N];
    const int nx = L.nx, ny = L.ny, n = L.nx * L.ny * L.nz;
    const int tid = threadIdx.x, tr = tid >> 5, tc = tid & 31, lane = tid & 63;
    double m[A][B];
#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int r = tr + 16 * a;
        const int i = r % nx + 1, j = (r / nx) % ny + 1, k = r / (nx * ny) + 1;
        const long long c = (long long)i + (long long)L.sy * j + L.sz * k;
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int q = tc + 32 * b;
            double v = 0.0;
            if (r < n && q < n) {
                if (q == r) v = S.st[ST_C][c];
                if (i > 1 && q == r - 1) v = S.st[ST_XM][c];
                if (i < nx && q == r + 1) v = S.st[ST_XP][c];
                if (j > 1 && q == r - nx) v = S.st[ST_YM][c];
                if (j < ny && q == r + nx) v = S.st[ST_YP][c];
                if (k > 1 && q == r - nx * ny) v = S.st[ST_ZM][c];
                if (k < L.nz && q == r + nx * ny) v = S.st[ST_ZP][c];
            }
            m[a][b] = v;
        }
    }
    if (tid < n) {
        // column tid: its diagonal, and its neighbours' entries for this cell
        const int i = tid % nx + 1, j = (tid / nx) % ny + 1, k = tid / (nx * ny) + 1;
        const long long c = (long long)i + (long long)L.sy * j + L.sz * k;
        double v = fabs(S.st[ST_C][c]);
        if (i > 1) v = fmax(v, fabs(S.st[ST_XP][c - 1]));
        if (i < nx) v = fmax(v, fabs(S.st[ST_XM][c + 1]));
        if (j > 1) v = fmax(v, fabs(S.st[ST_YP][c - L.sy]));
        if (j < ny) v = fmax(v, fabs(S.st[ST_YM][c + L.sy]));
        if (k > 1) v = fmax(v, fabs(S.st[ST_ZP][c - L.sz]));
        if (k < L.nz) v = fmax(v, fabs(S.st[ST_ZM][c + L.sz]));
        floor_of[tid] = kPivotFloor * v;
    }
    unsigned used = 0;   // bit t: row lane + 64 t has been a pivot row
    bool bad = false;
#pragma unroll
    for (int KB = 0; KB < B; ++KB) {
        for (int kc = 0; kc < 32; ++kc) {
            const int kk = 32 * KB + kc, buf = kc & 1;
            if (kk >= n) break;
            if (tc == kc) {
#pragma unroll
                for (int a = 0; a < A; ++a) {
                    scol[buf][tr + 16 * a] = m[a][KB];
                    m[a][KB] = 0.0;
                }
            }
            __syncthreads();
            unsigned long long key = 0;
#pragma unroll
            for (int t = 0; t < (N + 63) / 64; ++t) {
                const int r = lane + 64 * t;
                if (r < n && !((used >> t) & 1)) {
                    const double v = fabs(scol[buf][r]);
                    const unsigned long long bits = v == v ? __builtin_bit_cast(unsigned long long, v) : 0;
                    const unsigned long long w = (bits & ~0xffull) | (unsigned)(255 - r);
                    key = w > key ? w : key;
                }
            }
            key = dpp_max<0x111, 0xf>(key);   // row_shr 1, 2, 4, 8
            key = dpp_max<0x112, 0xf>(key);
            key = dpp_max<0x114, 0xf>(key);
            key = dpp_max<0x118, 0xf>(key);
            key = dpp_max<0x142, 0xa>(key);   // row_bcast 15, 31
            key = dpp_max<0x143, 0xc>(key);
            const unsigned klo = __builtin_amdgcn_readlane((int)key, 63);
            const unsigned khi = __builtin_amdgcn_readlane((int)(key >> 32), 63);
            // (an unused row below n always exists, so p < n)
            const int p = 255 - (int)(klo & 0xffu);
            if ((p & 63) == lane) used |= 1u << (p >> 6);
            const double piv = scol[buf][p];
            if (!(fabs(piv) > floor_of[kk])) bad = true;
            const int pr = p & 15, pa = p >> 4;
            if (tr == pr) {
#pragma unroll
                for (int a = 0; a < A; ++a) {
                    if (a == pa) {
#pragma unroll
                        for (int b = 0; b < B; ++b) {
                            srow[buf][tc + 32 * b] = m[a][b];
                            m[a][b] = 0.0;
                        }
                    }
                }
            }
            if (tid == 0) {
                perm[kk] = p;
                pos[p] = kk;
            }
            __syncthreads();
            // the pivot row becomes rk (0 - (-1) rk), every other row loses
            // its column entry times rk; column kk itself was set to zero
            const double inv = 1.0 / piv;
            double rk[B];
#pragma unroll
            for (int b = 0; b < B; ++b) rk[b] = ((b == KB && tc == kc) ? 1.0 : srow[buf][tc + 32 * b]) * inv;
#pragma unroll
            for (int a = 0; a < A; ++a) {
                const double f = (tr == pr && a == pa) ? -1.0 : scol[buf][tr + 16 * a];
#pragma unroll
                for (int b = 0; b < B; ++b) m[a][b] = fma(-f, rk[b], m[a][b]);
            }
        }
    }
    // row r holds the inverse's row pos[r]; column c belongs to row perm[c] of A
#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int r = tr + 16 * a;
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int q = tc + 32 * b;
            if (r < n && q < n) {
                Ainv[(long long)pos[r] * n + perm[q]] = m[a][b];
                if (AinvT) AinvT[(long long)perm[q] * n + pos[r]] = m[a][b];
            }
        }
    }
    if (tid == 0 && status) *status = bad ? -1 : 0;
}

// the same inverse with the matrix in global memory, for kInvRegsN < n
__global__ void __launch_bounds__(kDenseThreads) k_dense_inverse(Lev<double> L, RowArrays S, double *gwork, double *Ainv)
{
    __shared__ double col[kBottomMaxDense];
    __shared__ int perm[kBottomMaxDense];
    __shared__ double rv[kDenseThreads / 64];
    __shared__ int ri[kDenseThreads / 64];
    __shared__ int piv;
    const int nx = L.nx, ny = L.ny, n = L.nx * L.ny * L.nz;
    const int tid = threadIdx.x, nt = blockDim.x;
    const long long nn = (long long)n * n;
    double *const M = gwork;
    for (long long q = tid; q < nn; q += nt) M[q] = 0.0;
    __syncthreads();
    for (int r = tid; r < n; r += nt) {
        const int i = r % nx + 1, j = (r / nx) % ny + 1, k = r / (nx * ny) + 1;
        const long long c = (long long)i + (long long)L.sy * j + L.sz * k;
        double *row = M + (long long)r * n;
        row[r] = S.st[ST_C][c];
        if (i > 1) row[r - 1] = S.st[ST_XM][c];
        if (i < nx) row[r + 1] = S.st[ST_XP][c];
        if (j > 1) row[r - nx] = S.st[ST_YM][c];
        if (j < ny) row[r + nx] = S.st[ST_YP][c];
        if (k > 1) row[r - nx * ny] = S.st[ST_ZM][c];
        if (k < L.nz) row[r + nx * ny] = S.st[ST_ZP][c];
    }
    __syncthreads();
    for (int kk = 0; kk < n; ++kk) {
        // pivot: the largest |M[r][kk]|, r >= kk, lowest r on ties
        double best = -1.0;
        int bi = kk;
        for (int r = kk + tid; r < n; r += nt) {
            const double v = fabs(M[(long long)r * n + kk]);
            if (v > best) best = v, bi = r;
        }
        for (int off = 32; off > 0; off >>= 1) {
            const double ov = __shfl_down(best, off, 64);
            const int oi = __shfl_down(bi, off, 64);
            if (ov > best || (ov == best && oi < bi)) best = ov, bi = oi;
        }
        if ((tid & 63) == 0) rv[tid >> 6] = best, ri[tid >> 6] = bi;
        __syncthreads();
        if (tid == 0) {
            double b = rv[0];
            int p = ri[0];
            for (int w = 1; w < nt / 64; ++w)
                if (rv[w] > b || (rv[w] == b && ri[w] < p)) b = rv[w], p = ri[w];
            piv = p;
            perm[kk] = p;
        }
        __syncthreads();
        const int p = piv;
        double *rk = M + (long long)kk * n;
        if (p != kk) {
            double *rp = M + (long long)p * n;
            for (int q = tid; q < n; q += nt) {
                const double t = rk[q];
                rk[q] = rp[q];
                rp[q] = t;
            }
            __syncthreads();
        }
        const double inv = 1.0 / rk[kk];
        __syncthreads();
        // pivot row: M[kk][kk] = 1, then the row times 1 / pivot
        for (int q = tid; q < n; q += nt) rk[q] = (q == kk ? 1.0 : rk[q]) * inv;
        // the pivot column of the other rows, before the update
        for (int r = tid; r < n; r += nt) col[r] = M[(long long)r * n + kk];
        __syncthreads();
        // rows over the waves, columns over the lanes (no index division)
        for (int r = tid >> 6; r < n; r += nt >> 6) {
            if (r == kk) continue;
            const double f = col[r];
            double *row = M + (long long)r * n;
            for (int cidx = tid & 63; cidx < n; cidx += 64) row[cidx] = (cidx == kk ? 0.0 : row[cidx]) - f * rk[cidx];
        }
        __syncthreads();
    }
    // undo the row swaps as column swaps, last first
    for (int kk = n - 1; kk >= 0; --kk) {
        const int p = perm[kk];
        if (p != kk) {
            for (int r = tid; r < n; r += nt) {
                double *row = M + (long long)r * n;
                const double t = row[kk];
                row[kk] = row[p];
                row[p] = t;
            }
        }
        __syncthreads();
    }
    for (long long q = tid; q < nn; q += nt) Ainv[q] = M[q];
}

}  // namespace mps

namespace mps {

// dB/dx of the Bernoulli function, B'(x) = B(x) (1 - B(-x)) / x, with its
// Taylor series near 0 (B' = -1/2 + x/6 - x^3/180).
__device__ __forceinline__ double bernoulli_prime(double x)
{
    if (fabs(x) < 1e-3) {
        const double x2 = x * x;
        return -0.5 + x * (1.0 / 6.0 - x2 * (1.0 / 180.0));
    }
    return bernoulli(x) * (1.0 - bernoulli(-x)) / x;
}

// d(wL)/d(c) and d(wR)/d(c) of a face's flux weights with respect to the
// face velocity c = (cL + cR)/2 (SG: dwL/dc = -B'(-Pe), dwR/dc = -B'(Pe);
// upwind: the flux is c u_upwind); for vanishing D the SG weights are the
// upwind ones with the cell velocities, returned through dL/dR per cell.
template <int FLUX>
__device__ __forceinline__ void flux_dc(double cL, double cR, double DL, double DR, double d, double uL, double uR,
                                        double &g_face, double &g_L, double &g_R)
{
    const double ch = 0.5 * (cL + cR);
    g_face = 0.0;
    g_L = 0.0;
    g_R = 0.0;
    if (FLUX == MPS_FLUX_UPWIND_K) {
        g_face = ch > 0.0 ? uL : uR;
        return;
    }
    const double eps = 1e-10;
    const double Dh = 2.0 * DL * DR / (DL + DR + eps);
    if (fabs(Dh) < eps) {
        const double sgn = ch <= 0.0 ? -1.0 : 1.0;
        g_L = 0.5 * (1.0 + sgn) * uL;
        g_R = 0.5 * (1.0 - sgn) * uR;
        return;
    }
    const double Pe = ch * d / Dh;
    g_face = -bernoulli_prime(-Pe) * uL - bernoulli_prime(Pe) * uR;
}

// Velocity sensitivity of the adjoint pairing:  g_v(c) = -d(lam^T A(v) x)/dv(c)
// for the three cell velocity components, i.e. the gradient of a scalar J
// through x = A(v)^-1 b once lam = A^-T dJ/dx. Each face couples its two
// cells through the face velocity (v_L + v_R)/2 and the flux pairing
// (lam_L/w_L - lam_R/w_R) F; the boundary rows add their convective terms.
// Every cell evaluates both of its faces, so no atomics are needed.
template <int OP, int FLUX>
__global__ void __launch_bounds__(kBlock) k_velocity_grad(Lev<double> L, const double *__restrict__ lam,
                                                         const double *__restrict__ x, double *gx, double *gy,
                                                         double *gz)
{
    int i, j, k;
    long long c;
    if (!cell_of(L, i, j, k, c)) return;
    const double *vel[3] = {L.vx, L.vy, L.vz};
    const long long s[3] = {1, L.sy, L.sz};
    const int idx[3] = {i, j, k};
    const int nn[3] = {L.nx, L.ny, L.nz};
    const double h[3] = {L.dx, L.dy, L.dz};
    const double ai[3] = {L.ax, L.ay, L.az};
    const double ab[3] = {L.axb, L.ayb, L.azb};
    double *out[3] = {gx, gy, gz};
    const long long n = (long long)(i - 1) + (long long)L.nx * ((j - 1) + (long long)L.ny * (k - 1));
    for (int dim = 0; dim < 3; ++dim) {
        double g = 0.0;
        const double vc = vel[dim] ? vel[dim][c] : 0.0;
        auto abv_of = [&](int ii) {
            const bool edge = ii == 1 || ii == nn[dim];
            return (OP == OP_ALIGNED && edge) ? ab[dim] : ai[dim];
        };
        if (idx[dim] > 1) {  // face (m | c)
            const long long m = c - s[dim];
            double gf, gl, gr;
            flux_dc<FLUX>(vel[dim] ? vel[dim][m] : 0.0, vc, L.D[m], L.D[c], h[dim], x[m], x[c], gf, gl, gr);
            const double pair = lam[m] * abv_of(idx[dim] - 1) - lam[c] * abv_of(idx[dim]);
            g += pair * (0.5 * gf + gr);
        }
        if (idx[dim] < nn[dim]) {  // face (c | p)
            const long long p = c + s[dim];
            double gf, gl, gr;
            flux_dc<FLUX>(vc, vel[dim] ? vel[dim][p] : 0.0, L.D[c], L.D[p], h[dim], x[c], x[p], gf, gl, gr);
            const double pair = lam[c] * abv_of(idx[dim]) - lam[p] * abv_of(idx[dim] + 1);
            g += pair * (0.5 * gf + gl);
        }
        // boundary rows: DIRC upwind outflow and ZGRD convection
        // (discretepde.f90:810-828 and the + face copy)
        const double abv = abv_of(idx[dim]);
        const double hh = OP == OP_REF ? 1.0 / h[dim] : abv;
        if (idx[dim] == 1) {
            const int code = L.bc[2 * dim];
            if ((code == BC_DIRC && vc < 0.0) || code == BC_ZGRD) g += lam[c] * (-hh) * x[c];
        }
        if (idx[dim] == nn[dim]) {
            const int code = L.bc[2 * dim + 1];
            if ((code == BC_DIRC && vc > 0.0) || code == BC_ZGRD) g += lam[c] * hh * x[c];
        }
        out[dim][n] = -g;
    }
}

}  // namespace mps
