// Field passes of the multi-species discharge step (mps3d_amd/discharge.py):
// ghosted copies for the solver, the charge density, and everything between
// the Poisson solve and the species solves, on a stream of the caller's.
//
// All of it is streaming work. Written with one tensor operation per
// arithmetic operator a step of five species at 129^3 made some 80 passes
// over 17 MB fields; here the field, the mean energy, the rates and every
// right-hand side come from one pass that reads each input and writes each
// output once: that step went from 7.66 to 7.07 ms, a glow step at 128^3 from
// 7.37 to 6.65. The arithmetic is the operators',
// in their order and without contraction (a division by a number is the
// product with its reciprocal, as those operators take it).
#pragma once

#include <hip/hip_runtime.h>

#include "mps3d.h"

namespace mps {

constexpr int kDisX = 64, kDisY = 4;

// k fields (blockIdx.z / planes) of the interior copied into zero-ghosted
// ones, times scale. Three fields at 129^3 take 30 us (3.5 TB/s), the same by a
// fill and a strided copy each 58.
struct PadSet {
    const double *src[MPS_PAD_FIELDS];
    double *dst;
};
__global__ void __launch_bounds__(kDisX *kDisY) k_pad_fields(PadSet P, int nx, int ny, int nz, double scale)
{
    const int i = blockIdx.x * kDisX + threadIdx.x, j = blockIdx.y * kDisY + threadIdx.y;
    const int f = blockIdx.z / (nz + 2), k = blockIdx.z - f * (nz + 2);
    if (i >= nx + 2 || j >= ny + 2) return;
    double v = 0.0;
    if (i >= 1 && i <= nx && j >= 1 && j <= ny && k >= 1 && k <= nz)
        v = scale * P.src[f][(i - 1) + (long long)nx * ((j - 1) + (long long)ny * (k - 1))];
    P.dst[i + (long long)(nx + 2) * (j + (long long)(ny + 2) * blockIdx.z)] = v;
}

// right-hand side of the potential: coef * sum of the charges, and the
// electrode potentials in the first and last plane (DIRC rows of weight w)
__global__ void __launch_bounds__(kDisX *kDisY) k_charge_rhs(mps_discharge P, double *__restrict__ rhs, int nx, int ny, int nz)
{
    const int i = blockIdx.x * kDisX + threadIdx.x, j = blockIdx.y * kDisY + threadIdx.y, k = blockIdx.z;
    if (i >= nx || j >= ny) return;
    const long long q = i + (long long)nx * j, c = q + (long long)nx * ny * k;
    double rho = 0.0;
#pragma unroll
    for (int s = 0; s < MPS_DIS_SPECIES; ++s)
        if (s < P.nspecies && P.charge[s] != 0.0) rho = rho + P.charge[s] * P.dens[s][c];
    double r = P.rho_coef * rho;
    if (k == 0) r = r + (P.wall_weight * P.eps_r[c]) * P.lo[q];
    else if (k == nz - 1) r = r + (P.wall_weight * P.eps_r[c]) * P.hi[q];
    rhs[c] = r;
}

// The field E = -grad phi with its boundary rules, the mean electron energy,
// the reaction rates, and the right-hand side of every species and of the
// electron energy, from the old state. 79 us for five species at 129^3 (309
// MB, 3.9 TB/s), 38 us for two species and the energy at 128^3.
__global__ void __launch_bounds__(kDisX *kDisY) k_discharge_rhs(mps_discharge P, int nx, int ny, int nz)
{
    const int i = blockIdx.x * kDisX + threadIdx.x, j = blockIdx.y * kDisY + threadIdx.y, k = blockIdx.z;
    if (i >= nx || j >= ny) return;
    const long long sy = nx, sz = (long long)nx * ny, q = i + sy * j, c = q + sz * k;
    const double *phi = P.phi;
    const double u = phi[c], inv2h = 1.0 / (2.0 * P.h);
    const double xm = i > 0 ? phi[c - 1] : u, xp = i < nx - 1 ? phi[c + 1] : u;
    const double ym = j > 0 ? phi[c - sy] : u, yp = j < ny - 1 ? phi[c + sy] : u;
    const double zm = k > 0 ? phi[c - sz] : 2.0 * P.lo[q] - u;
    const double zp = k < nz - 1 ? phi[c + sz] : 2.0 * P.hi[q] - u;
    double n[MPS_DIS_SPECIES];
#pragma unroll
    for (int s = 0; s < MPS_DIS_SPECIES; ++s) n[s] = s < P.nspecies ? P.dens[s][c] : 0.0;
    const double neps = P.energy ? P.neps[c] : 0.0;
    const double ex = -(xp - xm) * inv2h, ey = -(yp - ym) * inv2h, ez = -(zp - zm) * inv2h;
    const long long nc = sz * nz;
    P.E[c] = ex;
    P.E[c + nc] = ey;
    P.E[c + 2 * nc] = ez;
    const double e2 = ex * ex + ey * ey + ez * ez;
    double ne = 0.0;
#pragma unroll
    for (int s = 0; s < MPS_DIS_SPECIES; ++s)
        if (s == P.electron) ne = n[s];
    double eb;
    if (P.energy) {
        eb = neps / ne;   // (a NaN stays one)
        eb = eb < 0.05 ? 0.05 : eb > 500.0 ? 500.0 : eb;
    } else {
        eb = P.eps0 * (1.0 + sqrt(e2 + 1e-30) * (1.0 / P.eps_ref));
    }
    const double Te = (2.0 / 3.0) * eb;
    const double ieb = 1.0 / eb;
    double R[MPS_DIS_REACTIONS];
#pragma unroll
    for (int r = 0; r < MPS_DIS_REACTIONS; ++r) {
        R[r] = 0.0;
        if (r >= P.nreactions) continue;
        double v = P.rate[r];
        if (P.arrhenius[r]) v = v * exp(ieb * -P.ea[r]);
        for (int m = 0; m < P.order[r]; ++m) {
            const int a = P.reactant[r][m];
            double f = P.gas;
#pragma unroll
            for (int s = 0; s < MPS_DIS_SPECIES; ++s)
                if (s == a) f = n[s];
            v = v * f;
        }
        R[r] = v;
    }
    const double idt = 1.0 / P.dt, ih = 1.0 / P.h;
    const bool plate = k == 0 || k == nz - 1;
    const double ce = sqrt(P.cbar_num * Te * (1.0 / P.cbar_den));   // electrons' thermal speed
    double qe = 0.0;                                                // and outflow
#pragma unroll
    for (int s = 0; s < MPS_DIS_SPECIES; ++s) {
        if (s >= P.nspecies) continue;
        double S = 0.0;
#pragma unroll
        for (int r = 0; r < MPS_DIS_REACTIONS; ++r)
            if (r < P.nreactions && P.nu[s][r] != 0.0) S = S + P.nu[s][r] * R[r];
        double b = n[s] * idt + S;
        if (P.outflow[s]) {
            const double qs = plate ? 0.25 * n[s] * (s == P.electron ? ce : P.cbar[s]) * ih : 0.0;
            b = b - qs;
            if (s == P.electron) qe = qs;
        }
        P.rhs[c + nc * s] = b;
    }
    if (P.energy) {
        double loss = P.elastic * ne * (Te - P.T_gas);
#pragma unroll
        for (int r = 0; r < MPS_DIS_REACTIONS; ++r)
            if (r < P.nreactions && P.loss[r] != 0.0) loss = loss + P.loss[r] * R[r];
        double b = neps * idt + P.mu_e * ne * e2 - loss;
        bool flow = false;
#pragma unroll
        for (int s = 0; s < MPS_DIS_SPECIES; ++s)
            if (s == P.electron) flow = P.outflow[s] != 0;
        if (flow) b = b - 2.0 * Te * qe;
        P.rhs[c + nc * P.nspecies] = b;
    }
}

}  // namespace mps
