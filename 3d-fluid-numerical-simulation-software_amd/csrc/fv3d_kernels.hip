// HIP kernels of the LU-SGS iteration for gfx950.
//
// One launch per stage covers every block of the mesh through a work list, so
// multi-block meshes cost no more launches than a single block.  Reductions
// (residual norm, section integrals) are two-pass with a fixed summation order
// and therefore deterministic run to run.
#include "fv3d_kernels.h"

#include <math.h>

namespace fv3d {

// ===================================================================== BC
// One thread per patch face.  Inlet (source/BndCondInlet.cpp:7-127), general
// and centrifugal outlet (source/BndCondOutlet.cpp:116-305), no-slip wall
// (source/BndCondWall.cpp:20-284).  Writes ghost cells of Q/W and the two
// Dummy layers of the patch side.
__device__ static void set_dummies(BlockRef B, int s, int a, int b, const double cv[5], const double pv[6])
{
    for (int l = 1; l <= kND; ++l) {
        for (int c = 0; c < 5; ++c) *dummy_ptr(B, s, l, c, a, b) = cv[c];
        for (int c = 0; c < 6; ++c) *dummy_ptr(B, s, l, 5 + c, a, b) = pv[c];
    }
}

// The pitch-angle sign of each periodic patch's block, updated in table order
// (source/BndCondInteriorPeriodic.cpp:54-59): patches that share a block see
// each other's flips.  How often a patch's block has flipped by then is known
// (PeriodicDev::odd), so one workgroup takes the patches side by side; one
// thread walking them was 0.3 us each, the tail of the boundary kernel.
__device__ static void periodic_flip(PeriodicDev *per, int nper, int *pitch_sign)
{
    for (int p = threadIdx.x; p < nper; p += blockDim.x) {
        const int s = pitch_sign[per[p].block];
        per[p].sign = per[p].odd ? -s : s;
    }
    __syncthreads();
    for (int p = threadIdx.x; p < nper; p += blockDim.x)
        if (per[p].last) pitch_sign[per[p].block] = per[p].sign;
}

// Ghost cells and Dummy layers of boundary item t (inlet, outlet, wall).
__device__ static void bc_item(const BlockDev *__restrict__ blocks, const PatchDev *__restrict__ patches, int npatch,
                               const long *__restrict__ pstart, const Gas &g, const ScalarsDev *__restrict__ sc, long t)
{
    if (t >= pstart[npatch]) return;
    const int q = find_range(pstart, npatch, t);
    const PatchDev P = patches[q];
    BlockRef B = block_at(blocks, P.block);
    long r = t - pstart[q];
    int a = P.a0 + (int)(r / P.nb), b = P.b0 + (int)(r % P.nb);   // tangential cell indices
    const int d = P.dir, hi = P.hi;
    const int N = d == 0 ? B.IM : d == 1 ? B.JM : B.KM;
    // interior cell next to the face and the ghost cell behind it
    int ii, jj, kk, gi, gj, gk;
    int pi = hi ? N - 1 : 1, pg = hi ? N : 0;
    if (d == 0) { ii = pi; gi = pg; jj = gj = a; kk = gk = b; }
    else if (d == 1) { jj = pi; gj = pg; ii = gi = a; kk = gk = b; }
    else { kk = pi; gk = pg; ii = gi = a; jj = gj = b; }
    const long xi = cidx(B, ii, jj, kk), xg = cidx(B, gi, gj, gk);
    const long box = B.box;
    const int s = 2 * d + hi;
    const double Gamma = g.gamma, Rgas = g.rgas;
    double cv[5], pv[6];
    if (P.kind == 0) {
        // inlet: K faces only
        if (d != 2) return;
        const int kf = hi ? N : 1;
        const long xf = cidx(B, ii, jj, kf);
        double Sx = B.fS[2][xf], Sy = B.fS[2][box + xf], Sz = B.fS[2][2 * box + xf];
        double n_m = sqrt(Sx * Sx + Sy * Sy + Sz * Sz);
        double uvel = B.W[1 * box + xi], vvel = B.W[2 * box + xi], wvel = B.W[3 * box + xi];
        double vdn = uvel * Sx / n_m + vvel * Sy / n_m + wvel * Sz / n_m;
        if (!hi) vdn = F32C(-1.0) * vdn;
        const double *A = g.inlet_dir;
        double Vn_m = sqrt(A[0] * A[0] + A[1] * A[1] + A[2] * A[2]);
        double c_d = sqrt(Gamma * Rgas * B.W[5 * box + xi]);
        double V2_d = uvel * uvel + vvel * vvel + wvel * wvel;
        double costh = F32C(-1.0) * vdn / sqrt(V2_d);
        double c_02 = c_d * c_d + (Gamma - F32C(1.0)) * V2_d / F32C(2.0);
        double R_minus = vdn - F32C(2.0) * c_d / (Gamma - F32C(1.0));
        double meduA = (-R_minus * (Gamma - F32C(1.0))) / ((Gamma - F32C(1.0)) * costh * costh + F32C(2.0));
        double meduB = sqrt(c_02 * ((Gamma - F32C(1.0)) * costh * costh + F32C(2.0)) / (Gamma - F32C(1.0)) /
                                (R_minus * R_minus) - (Gamma - F32C(1.0)) / F32C(2.0));
        double c_b = meduA * (F32C(1.0) + costh * meduB);
        double Ttin = g.tt_in, Ptin = g.pt_in;
        double TempBC = Ttin * (c_b * c_b / c_02);
        if (TempBC > Ttin) TempBC = F32C(0.99) * Ttin;
        double PressBC = Ptin * pow(TempBC / Ttin, Gamma / (Gamma - F32C(1.0)));
        double DensBC = PressBC / Rgas / TempBC;
        double VBC = sqrt(F32C(2.0) * Gamma / (Gamma - 1) * Rgas * (Ttin - TempBC));
        double u = VBC * A[0] / Vn_m, v = VBC * A[1] / Vn_m, w = VBC * A[2] / Vn_m;
        double V2 = u * u + v * v + w * w;
        double ener = PressBC / DensBC / (Gamma - F32C(1.0)) + V2 / F32C(2.0);
        pv[0] = DensBC; pv[1] = u; pv[2] = v; pv[3] = w; pv[4] = PressBC; pv[5] = TempBC;
        cv[0] = DensBC; cv[1] = DensBC * u; cv[2] = DensBC * v; cv[3] = DensBC * w; cv[4] = DensBC * ener;
        if (B.ev) B.ev[xg] = g.ev_ratio * F32C(1.0);   // source/BndCondInlet.cpp:104-105
    } else if (P.kind == 1) {
        // general / centrifugal outlet, K faces only (the radial-equilibrium
        // outlet is k_bc_axial's)
        if (d != 2 || P.axial) return;
        const int kf = hi ? N : 1;
        const long xf = cidx(B, ii, jj, kf);
        double s_ = B.fs[2][xf];
        double nx = B.fS[2][xf] / s_, ny = B.fS[2][box + xf] / s_, nz = B.fS[2][2 * box + xf] / s_;
        double d0 = B.W[xi], u0 = B.W[box + xi], v0 = B.W[2 * box + xi], w0 = B.W[3 * box + xi];
        double p0 = B.W[4 * box + xi], T0 = B.W[5 * box + xi];
        double Pout = sc[P.inst].p_out;
        double dens0 = d0;
        double c0 = sqrt(Gamma * Rgas * T0);
        double Vn = u0 * nx + v0 * ny + w0 * nz;
        double Ma_n = Vn / c0;
        if (P.centrifugal || Ma_n <= 1.0) {
            pv[4] = Pout;
            pv[0] = d0 + (Pout - p0) / c0 / c0;
            pv[1] = u0 + nx * (p0 - Pout) / dens0 / c0;
            pv[2] = v0 + ny * (p0 - Pout) / dens0 / c0;
            pv[3] = w0 + nz * (p0 - Pout) / dens0 / c0;
        } else {
            pv[4] = p0; pv[0] = d0; pv[1] = u0; pv[2] = v0; pv[3] = w0;
        }
        pv[5] = pv[4] / pv[0] / Rgas;
        double V2 = pv[1] * pv[1] + pv[2] * pv[2] + pv[3] * pv[3];
        double ener = pv[4] / pv[0] / (Gamma - F32C(1.0)) + V2 / F32C(2.0);
        cv[0] = pv[0]; cv[1] = pv[0] * pv[1]; cv[2] = pv[0] * pv[2]; cv[3] = pv[0] * pv[3]; cv[4] = pv[0] * ener;
        if (B.ev) B.ev[xg] = B.ev[xi];   // source/BndCondOutlet.cpp:180-181, 282-283
    } else {
        // no-slip wall: mirror the relative velocity about the wall velocity
        const int f = hi ? N : 1;
        const long xf = d == 0 ? cidx(B, f, jj, kk) : d == 1 ? cidx(B, ii, f, kk) : cidx(B, ii, jj, f);
        double x = B.fc[d][xf], y = B.fc[d][box + xf];
        double rot = P.rot;
        double Vwall_x = -rot * y, Vwall_y = rot * x;
        double Vin_x = B.W[box + xi] - Vwall_x, Vin_y = B.W[2 * box + xi] - Vwall_y, Vin_z = B.W[3 * box + xi] - F32C(0.0);
        double Vout_x = F32C(0.0) - Vin_x, Vout_y = F32C(0.0) - Vin_y, Vout_z = F32C(0.0) - Vin_z;
        pv[0] = B.W[xi];
        pv[1] = Vout_x + Vwall_x;
        pv[2] = Vout_y + Vwall_y;
        pv[3] = Vout_z + F32C(0.0);
        pv[4] = B.W[4 * box + xi];
        pv[5] = B.W[5 * box + xi];
        cv[0] = B.Q[xi];
        cv[1] = pv[1] * cv[0];
        cv[2] = pv[2] * cv[0];
        cv[3] = pv[3] * cv[0];
        cv[4] = B.Q[4 * box + xi];
        for (int c = 0; c < 5; ++c) B.Q[c * box + xg] = cv[c];
        for (int c = 0; c < 6; ++c) B.W[c * box + xg] = pv[c];
        if (B.ev) B.ev[xg] = F32C(0.0);   // source/BndCondWall.cpp:104-107
        double cd[5], pd[6];
        for (int c = 0; c < 5; ++c) cd[c] = (cv[c] + B.Q[c * box + xi]) * 0.5;
        for (int c = 0; c < 6; ++c) pd[c] = 0.5 * (pv[c] + B.W[c * box + xi]);
        set_dummies(B, s, a, b, cd, pd);
        return;
    }
    for (int c = 0; c < 5; ++c) B.Q[c * box + xg] = cv[c];
    for (int c = 0; c < 6; ++c) B.W[c * box + xg] = pv[c];
    set_dummies(B, s, a, b, cv, pv);
}

// One transfer of source/ShadowOutIn.cpp: Trans rotates the momentum and the
// velocity about z by dr when dr != 0 (lines 188-199).
__device__ static void exchange_item(const BlockDev *__restrict__ blocks, const ExchDev *__restrict__ el, long n,
                                     const PeriodicDev *per, long t)
{
    if (t >= n) return;
    const ExchDev e = el[t];
    // One (source block, target block, side) of the wave's lanes after the other,
    // nearly always one in all: what the block tables hold then comes through
    // scalar loads.
    for (unsigned long long left = __builtin_amdgcn_ballot_w64(true); left;) {
        const int l = __builtin_ctzll(left);
        const int sb = __builtin_amdgcn_readlane(e.src_block, l), db = __builtin_amdgcn_readlane(e.dst_block, l),
                  side = __builtin_amdgcn_readlane(e.side, l);
        const bool in = e.src_block == sb && e.dst_block == db && e.side == side;
        left &= ~__builtin_amdgcn_ballot_w64(in);
        if (!in) continue;
        BlockRef A = block_at(blocks, sb), B = block_at(blocks, db);
        double q[5], w[6];
        for (int c = 0; c < 5; ++c) q[c] = A.Q[c * A.box + e.src];
        for (int c = 0; c < 6; ++c) w[c] = A.W[c * A.box + e.src];
        if (e.rot) {
            const PeriodicDev &P = per[e.per];
            const bool pos = (e.rot == 1) == (P.sign > 0);   // dr = +delta or -delta
            const double cr = pos ? P.cs[0] : P.cs[2], sr = pos ? P.cs[1] : P.cs[3];
            const double qx = q[1], qy = q[2], ux = w[1], uy = w[2];
            q[1] = qx * cr - qy * sr;
            q[2] = qy * cr + qx * sr;
            w[1] = ux * cr - uy * sr;
            w[2] = uy * cr + ux * sr;
        }
        const long Dt = B.Dt[side];
        double *D = B.D[side] + (long)(e.layer - 1) * 11 * Dt + e.slot;
        for (int c = 0; c < 5; ++c) D[c * Dt] = q[c];
        for (int c = 0; c < 6; ++c) D[(5 + c) * Dt] = w[c];
        if (e.ghost >= 0) {
            for (int c = 0; c < 5; ++c) B.Q[c * B.box + e.ghost] = q[c];
            for (int c = 0; c < 6; ++c) B.W[c * B.box + e.ghost] = w[c];
            if (B.ev) B.ev[e.ghost] = A.ev[e.src];   // nu~ of the ghost layer only (source/ShadowOutIn.cpp:339-345)
        }
    }
}

// Boundary conditions: nbcg workgroups fill the ghost cells of inlets, outlets
// and walls, one updates the periodic signs where nflip patches need it, the
// others run the exchange.  Nothing here orders these against each other.  All three
// may come in one launch only if no transfer ends on a cell that a boundary
// patch fills too (or a radial-equilibrium outlet, which comes between the two)
// and no sign flips: launch_bc sees to that (bc_overlap, n_axial, nflip) and
// otherwise launches the fills with the signs first, then the exchange.  Both
// read interior cells only.  They are look-ups and one round of loads, bound by
// latency (on large K faces by the exchange's scattered lines): as two launches
// 25 us on a rotor-stator stage, 42 us on a batch of eight passages, 69 us on
// 2.54M cells; as one 18, 33 and 58 us.  A long exchange goes by itself again
// (kManyExch).  84 registers, five waves per SIMD: held to 64 for eight waves, the
// fills of a 16x512x512 channel took 62 us instead of 58, of 192x192x512 71 instead
// of 67, and the passages' exchanges 2 % more.
__global__ void __launch_bounds__(256)
k_boundary(const BlockDev *__restrict__ blocks, const PatchDev *__restrict__ patches, int npatch,
           const long *__restrict__ pstart, int nbcg, Gas g, const ScalarsDev *__restrict__ sc,
           const ExchDev *__restrict__ el, long nexch, PeriodicDev *per, int nflip, int *pitch_sign)
{
    const int b = blockIdx.x;
    if (b < nbcg) bc_item(blocks, patches, npatch, pstart, g, sc, (long)b * 256 + threadIdx.x);
    else if (nflip > 0 && b == nbcg) periodic_flip(per, nflip, pitch_sign);
    else exchange_item(blocks, el, nexch, per, (long)(b - nbcg - (nflip > 0)) * 256 + threadIdx.x);
}

// CBndConds::BndCondOutlet_Axial (source/BndCondOutlet.cpp:7-114): static
// pressure in radial equilibrium, dp/dr = rho c_u^2 / r, fixed to Pout at
// i = (int)(0.5 IM) and integrated outwards along i on every j line; c_u is the
// area-weighted circumferential velocity of the last cell layer per i.  As in
// the reference it covers the whole K+ face of the block, reads the density of
// the ghost layer left by the previous application, and integrates towards
// the tip with the radii of the faces at KM-1.  One workgroup per patch: the
// per-i averages (serial over j, the reference's order), then one thread per
// j line, then the ghost cells and Dummy layers.
__global__ void __launch_bounds__(256) k_bc_axial(const BlockDev *__restrict__ blocks,
                                                  const PatchDev *__restrict__ patches, const int *__restrict__ list,
                                                  Gas g, const ScalarsDev *__restrict__ sc)
{
    __shared__ double cu[kAxialMaxI];
    const PatchDev P = patches[list[blockIdx.x]];
    if (P.dir != 2 || !P.hi) return;   // K+ faces only (source/BndCondOutlet.cpp:33-41)
    BlockRef B = block_at(blocks, P.block);
    const int IM = B.IM, JM = B.JM, KM = B.KM, k = KM - 1;
    const long box = B.box;
    const double *fc = B.fc[2], *fs = B.fs[2];
    const double Gamma = g.gamma, Rgas = g.rgas;
    for (int i = 1 + (int)threadIdx.x; i <= IM - 1; i += blockDim.x) {
        double c_u = 0.0, S_temp = 0.0;
        for (int j = 1; j <= JM - 1; ++j) {
            const long xc = cidx(B, i, j, k), xf = cidx(B, i, j, KM);
            const double th = atan(fc[box + xf] / fc[xf]);
            const double cu_temp = F32C(-1.0) * B.W[box + xc] * sin(th) + B.W[2 * box + xc] * cos(th);
            c_u = c_u + cu_temp * fs[xf];
            S_temp = S_temp + fs[xf];
        }
        cu[i] = c_u / S_temp;
    }
    __syncthreads();
    const int iref = (int)(0.5 * IM);
    const double Pout = sc[P.inst].p_out;
    auto rad = [&](int i, int j, int kk) {
        const long xf = cidx(B, i, j, kk);
        return sqrt(fc[xf] * fc[xf] + fc[box + xf] * fc[box + xf]);
    };
    double *p = B.W + 4 * box;
    for (int j = 1 + (int)threadIdx.x; j <= JM - 1; j += blockDim.x) {
        p[cidx(B, iref, j, KM)] = Pout;
        for (int i = iref - 1; i >= 1; --i) {
            const double rn = rad(i, j, KM), rn_1 = rad(i + 1, j, KM);
            const double dp_dr = B.Q[cidx(B, i, j, KM)] * cu[i] * cu[i] / rn;
            p[cidx(B, i, j, KM)] = p[cidx(B, i + 1, j, KM)] - dp_dr * (rn_1 - rn);
        }
        for (int i = iref + 1; i <= IM - 1; ++i) {
            const double rn_1 = rad(i, j, k), rn = rad(i - 1, j, k);
            const double dp_dr = B.Q[cidx(B, i, j, KM)] * cu[i] * cu[i] / rn;
            p[cidx(B, i, j, KM)] = p[cidx(B, i - 1, j, KM)] + dp_dr * (rn_1 - rn);
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < (IM - 1) * (JM - 1); e += blockDim.x) {
        const int i = 1 + e / (JM - 1), j = 1 + e % (JM - 1);
        const long xg = cidx(B, i, j, KM), xi = cidx(B, i, j, k);
        double cv[5], pv[6];
        for (int c = 0; c < 4; ++c) cv[c] = B.Q[c * box + xi];
        pv[0] = cv[0];
        pv[1] = B.W[box + xi]; pv[2] = B.W[2 * box + xi]; pv[3] = B.W[3 * box + xi];
        pv[4] = p[xg];
        pv[5] = pv[4] / Rgas / cv[0];
        const double V2 = pv[1] * pv[1] + pv[2] * pv[2] + pv[3] * pv[3];
        cv[4] = pv[4] / (Gamma - F32C(1.0)) + pv[0] * V2 / F32C(2.0);
        for (int c = 0; c < 5; ++c) B.Q[c * box + xg] = cv[c];
        for (int c = 0; c < 6; ++c) B.W[c * box + xg] = pv[c];
        if (B.ev) B.ev[xg] = B.ev[xi];   // source/BndCondOutlet.cpp:102-103
        set_dummies(B, 5, i, j, cv, pv);
    }
}

// Global time step of CTimeDiscr::TimeStep (source/TimeStep.cpp:64-86): the
// minimum over each block's cells, starting from 1E10 (the caller fills dtmin
// with its bits), then every cell of the block takes it and the LU-SGS
// diagonal is formed again from it.  Time steps are positive, so the bits
// order as the values.
__global__ void __launch_bounds__(256) k_dt_block_min(const BlockDev *__restrict__ blocks, const long *__restrict__ cstart,
                                                      int nblock, unsigned long long *__restrict__ dtmin)
{
    constexpr int kSlots = 16;
    __shared__ unsigned long long smin[kSlots];
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long t0 = (long)blockIdx.x * blockDim.x;
    const int n0 = t0 < cstart[nblock] ? find_range(cstart, nblock, t0) : nblock - 1;
    if (threadIdx.x < kSlots) smin[threadIdx.x] = ~0ull;
    __syncthreads();
    int n, i, j, k;
    if (cell_item(blocks, cstart, nblock, t, n, i, j, k)) {
        BlockRef B = block_at(blocks, n);
        const unsigned long long v = (unsigned long long)__double_as_longlong(B.dt[cidx(B, i, j, k)]);
        if (n - n0 < kSlots) atomicMin(&smin[n - n0], v);
        else atomicMin(dtmin + n, v);
    }
    __syncthreads();
    if (threadIdx.x < kSlots && n0 + (int)threadIdx.x < nblock && smin[threadIdx.x] != ~0ull)
        atomicMin(dtmin + n0 + threadIdx.x, smin[threadIdx.x]);
}

__global__ void __launch_bounds__(256) k_dt_global(const BlockDev *__restrict__ blocks, const long *__restrict__ cstart,
                                                   int nblock, Gas g, const unsigned long long *__restrict__ dtmin)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int n, i, j, k;
    if (!cell_item(blocks, cstart, nblock, t, n, i, j, k)) return;
    BlockRef B = block_at(blocks, n);
    const long box = B.box, x = cidx(B, i, j, k);
    const double dt = __longlong_as_double((long long)dtmin[n]);
    B.dt[x] = dt;
    double lvd[3] = {0.0, 0.0, 0.0};
    if (g.viscous)
        for (int d = 0; d < 3; ++d) lvd[d] = B.lamv[d * box + x];
    B.alpha[x] = B.vol[x] / dt + g.relax * (B.lamc[x] + B.lamc[box + x] + B.lamc[2 * box + x]) +
                 F32C(2.0) * (lvd[0] + lvd[1] + lvd[2]);
    if (B.alpha2)
        B.alpha2[x] = B.vol[x] / dt + g.relax * (B.lamc[x] + B.lamc[box + x] + B.lamc[2 * box + x]) +
                      F32C(3.0) * (lvd[0] + lvd[1] + lvd[2]);
}

// ======================================================= spectral + dt
// source/Spectral_curl_grad.cpp:9-42 and source/TimeStep.cpp:7-62, with the
// viscous spectral radii for Navier-Stokes (TimeStep.cpp:38-49).
__global__ void k_spectral_dt(const BlockDev *__restrict__ blocks, const long *__restrict__ cstart, int nblock, Gas g)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for_cell_item(blocks, cstart, nblock, t, [&](BlockRef B, int, int i, int j, int k) {
        const long box = B.box, x = cidx(B, i, j, k);
        const double Gamma = g.gamma, Rgas = g.rgas;
        double uvelr = B.W[box + x] + B.w_rot * B.cc[box + x];
        double vvelr = B.W[2 * box + x] - B.w_rot * B.cc[x];
        double wvelr = B.W[3 * box + x];
        double csoun = sqrt(Gamma * Rgas * B.W[5 * box + x]);
        double lam[3], eq[3];
        const long xn[3] = {x + B.si, x + B.sj, x + 1};
        for (int d = 0; d < 3; ++d) {
            const double *S = B.fS[d];
            double Sx = (S[x] + S[xn[d]]) * F32C(0.5);
            double Sy = (S[box + x] + S[box + xn[d]]) * F32C(0.5);
            double Sz = (S[2 * box + x] + S[2 * box + xn[d]]) * F32C(0.5);
            eq[d] = Sx * Sx + Sy * Sy + Sz * Sz;
            double CS = csoun * sqrt(eq[d]);
            lam[d] = fabs(uvelr * Sx + vvelr * Sy + wvelr * Sz) + CS;
            B.lamc[d * box + x] = lam[d];
        }
        int flag = *B.flag_low_dt;
        double dt_factor = flag == 0 ? F32C(1.0) : (double)(1.0f / (1.0f + (float)flag));
        double lc = lam[0] + lam[1] + lam[2];
        double lv = 0.0, lvd[3] = {0.0, 0.0, 0.0};
        if (g.viscous) {
            const double mue_lam = sutherland(g, B.W[5 * box + x]), mue_tur = B.mut ? B.mut[x] : 0.0, dens = B.W[x];
            const double a = (double)(4.0f / 3.0f) / dens, b = Gamma / dens;
            const double m = a > b ? a : b;
            for (int d = 0; d < 3; ++d) {
                lvd[d] = m * (mue_lam / g.pr_lam + mue_tur / g.pr_tur) * eq[d] / B.vol[x];
                B.lamv[d * box + x] = lvd[d];
            }
            lv = lvd[0] + lvd[1] + lvd[2];
        }
        double dt = dt_factor * (*B.cfl) * B.vol[x] / (lc + g.c_timestep * lv);
        B.dt[x] = dt;
        // diagonal of the LU-SGS operator (source/LU_SGS_Marching.cpp:76-77)
        B.alpha[x] = B.vol[x] / dt + g.relax * (lam[0] + lam[1] + lam[2]) + F32C(2.0) * (lvd[0] + lvd[1] + lvd[2]);
        // and of its nu~ equation (source/LU_SGS_Marching.cpp:81-82)
        if (B.alpha2)
            B.alpha2[x] = B.vol[x] / dt + g.relax * (lam[0] + lam[1] + lam[2]) + F32C(3.0) * (lvd[0] + lvd[1] + lvd[2]);
    });
}

// As a launch of its own for a TimeStep that no convective residual follows.
__global__ void k_dt_flag_decrement(const BlockDev *__restrict__ blocks, int nblock) { flag_decrement(blocks, nblock); }

// =================================================== convective residual
// Face flux of CSpaceDiscr::Upwind_Convective (source/Upwind_Convective.cpp:5-360)
// with the WallFlux override (source/WallFlux.cpp:70-175).
template <int MODE>
__device__ static void face_flux(BlockRef B, const Gas &g, int d, int i, int j, int k, double out[5])
{
    const long box = B.box;
    const int N = d == 0 ? B.IM : d == 1 ? B.JM : B.KM;
    const int p = d == 0 ? i : d == 1 ? j : k;
    const long xf = cidx(B, i, j, k);
    if (p == 1 || p == N) {
        const int s = 2 * d + (p == N);
        const int ta = d == 0 ? j : i, tb = d == 2 ? j : k;
        const long tix = (long)ta * B.Db[s] + tb;
        if (B.wmask[s] != nullptr && B.wmask[s][tix]) {
            const long xb = xf - (d == 0 ? B.si : d == 1 ? B.sj : 1);
            double wa[5], wb[5];
            for (int c = 0; c < 5; ++c) { wa[c] = B.W[c * box + xf]; wb[c] = B.W[c * box + xb]; }
            wall_face_core(g.gamma, wa, wb, B.fS[d][xf], B.fS[d][box + xf], B.fS[d][2 * box + xf], B.fc[d][xf],
                           B.fc[d][box + xf], B.wrot[s][tix], out);
            return;
        }
    }
    // four-cell stencil along d; cells outside [1, N-1] come from the Dummy
    // layers.  Characteristic reconstruction (any variable code other than
    // 100 and 200, source/UserInput.cpp:117-130) takes the conservative
    // stencil and the primitive variables of F and B.
    constexpr bool prim = MODE == 0, chr = MODE == 2;
    double st[4][5], wFB[2][6];
    const long dstride = d == 0 ? B.si : d == 1 ? B.sj : 1;
    const double *src = prim ? B.W : B.Q;
    for (int o = 0; o < 4; ++o) {
        int pc = p - 2 + o;
        if (pc >= 1 && pc <= N - 1) {
            long xc = xf + (long)(o - 2) * dstride;
            for (int c = 0; c < 5; ++c) st[o][c] = src[c * box + xc];
            if (chr && (o == 1 || o == 2))
                for (int c = 0; c < 6; ++c) wFB[o - 1][c] = B.W[c * box + xc];
        } else {
            int s = 2 * d + (pc >= N ? 1 : 0);
            int layer = pc < 1 ? 1 - pc : pc - (N - 1);
            int ta = d == 0 ? j : i, tb = d == 2 ? j : k;
            int c0 = prim ? 5 : 0;
            for (int c = 0; c < 5; ++c) st[o][c] = *dummy_ptr(B, s, layer, c0 + c, ta, tb);
            if (chr && (o == 1 || o == 2))
                for (int c = 0; c < 6; ++c) wFB[o - 1][c] = *dummy_ptr(B, s, layer, 5 + c, ta, tb);
        }
    }
    const long xd = d == 0 ? cidx(B, i, j + 1, k + 1) : d == 1 ? cidx(B, i + 1, j, k + 1) : cidx(B, i + 1, j + 1, k);
    // a non-rotating block skips the face centroid (its grid velocity is zero)
    double fcx = 0.0, fcy = 0.0;
    if (B.w_rot != 0.0) { fcx = B.fc[d][xf]; fcy = B.fc[d][box + xf]; }
    face_core<MODE>(g, st, wFB[0], wFB[1], B.fS[d][xf], B.fS[d][box + xf], B.fS[d][2 * box + xf], B.fs[d][xf], fcx, fcy,
              B.w_rot, B.node[xd] - B.node[xf], B.node[box + xd] - B.node[box + xf],
              B.node[2 * box + xd] - B.node[2 * box + xf], out);
}

// Tile of TI x TJ x TK cells per workgroup; every face of the tile is computed
// once into LDS, then each cell sums its six faces and subtracts the rotation
// source (source/ComputeAllBlockVars.cpp:85-118, 237-254).  Optionally stores
// the face fluxes for inspection.
//
// The face code is bound by FP64 issue, so what counts is how many times a wave
// runs it.  The tile's faces (about 3.5 per cell) are handed out 64 at a time,
// each group of one direction (so the direction and every array it selects is
// wave-uniform): 15 or 16 groups for every shape, at most four per wave.  With
// the faces handed out by cell (each thread its three low faces, the threads on
// the tile's upper edges the high ones) a wave ran the code six times, the last
// three with an eighth to a half of its lanes: 651 -> 494 us on a 2.54M-cell
// passage (4x4x16), 260 -> 201 us on a 1.05M-cell channel.  With one
// reconstruction per kernel the face code fits 128 registers and four waves per
// SIMD: 494 -> 467 us, 201 -> 188 us (the characteristic one needs 166 and
// keeps three).
// On a small grid the time is one workgroup's rounds of face code: with NT threads,
// as many as the registers allow, the groups take one round (two for the
// characteristic form) instead of four: 19 -> 12 us on 576 cells, 28.8 -> 26.3
// on 98k (384 tiles).  The kernel of 256 threads stays for the others: built for up to 1024
// it spills more and is 4 % slower on 1M cells.
template <int TI, int TJ, int TK, int MODE, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(MODE == 2 ? 3 : 4)))
k_convective(const BlockDev *__restrict__ blocks, const int4 *__restrict__ tiles, Gas g, int ndec, int store_faces,
             double *fI0, double *fJ0, double *fK0)
{
    if (blockIdx.x == 0) flag_decrement(blocks, ndec);
    constexpr int NFI = (TI + 1) * TJ * TK, NFJ = TI * (TJ + 1) * TK, NFK = TI * TJ * (TK + 1);
    constexpr int GI = (NFI + 63) / 64, GJ = (NFJ + 63) / 64, GK = (NFK + 63) / 64;   // groups per direction
    __shared__ double sI[5][TI + 1][TJ][TK];
    __shared__ double sJ[5][TI][TJ + 1][TK];
    __shared__ double sK[5][TI][TJ][TK + 1];
    const int4 tl = tiles[blockIdx.x];
    if (tl.x < 0) return;   // padding of the XCD-ordered tile list
    BlockRef B = block_at(blocks, tl.x);
    const int t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    // one copy of the face code in a rolled loop: a copy per direction (every
    // scheme and both fluxes) would crowd the instruction cache
#pragma nounroll
    for (int q = wave; q < GI + GJ + GK; q += NT / 64) {
        const int d = q < GI ? 0 : q < GI + GJ ? 1 : 2;
        const int f = (q - (d == 0 ? 0 : d == 1 ? GI : GI + GJ)) * 64 + lane;   // face number within its direction
        // place in the tile; the divisors are constants in each branch
        int a, b, c;
        if (d == 0) { c = f % TK; b = f / TK % TJ; a = f / (TK * TJ); }
        else if (d == 1) { c = f % TK; b = f / TK % (TJ + 1); a = f / (TK * (TJ + 1)); }
        else { c = f % (TK + 1); b = f / (TK + 1) % TJ; a = f / ((TK + 1) * TJ); }
        const int i = tl.y + a + 1, j = tl.z + b + 1, k = tl.w + c + 1;   // the face's higher cell
        if (a >= TI + (d == 0) || i > B.ni + (d == 0) || j > B.nj + (d == 1) || k > B.nk + (d == 2)) continue;
        double out[5];
        // gamma anew each time round: what depends on it alone is a few
        // instructions, but kept across the loop it takes the registers that the
        // face code then spills (1.03 GB moved instead of 0.78 on 2.54M cells,
        // 431 -> 393 us; 1.05M cells 159 -> 153).  On conservative variables it
        // gains 8 % with the Roe flux on 1.05M cells (166 -> 154) and 2 % on
        // 292k (64.5 -> 63.4), but costs 2 % with Steger-Warming there (61.3 -> 62.4):
        // the flux is a run-time choice of one kernel, so both get it.  The
        // characteristic form takes 156 registers instead of 168, the same time.
        Gas gl = g;
        asm volatile("" : "+s"(gl.gamma));
        face_flux<MODE>(B, gl, d, i, j, k, out);
        double *dst = (d == 0 ? &sI[0][0][0][0] : d == 1 ? &sJ[0][0][0][0] : &sK[0][0][0][0]) + f;
        const int n = d == 0 ? NFI : d == 1 ? NFJ : NFK;
        for (int e = 0; e < 5; ++e) dst[e * n] = out[e];
    }
    __syncthreads();
    if (t >= TI * TJ * TK) return;
    const int tk = t % TK, tj = (t / TK) % TJ, ti = t / (TK * TJ);
    const int i = tl.y + ti + 1, j = tl.z + tj + 1, k = tl.w + tk + 1;
    if (i > B.ni || j > B.nj || k > B.nk) return;
    const long box = B.box, x = cidx(B, i, j, k);
    const double w_rot = B.w_rot;
    const double vol = B.vol[x];
    const double dens = B.W[x], uvel = B.W[box + x], vvel = B.W[2 * box + x];
    double Qc[5] = {0.0, dens * (w_rot * vvel) * vol, F32C(-1.0) * dens * (w_rot * uvel) * vol, 0.0, 0.0};
    for (int c = 0; c < 5; ++c) {
        double s = sI[c][ti + 1][tj][tk] - sI[c][ti][tj][tk];
        s = s + sJ[c][ti][tj + 1][tk];
        s = s - sJ[c][ti][tj][tk];
        s = s + sK[c][ti][tj][tk + 1];
        s = s - sK[c][ti][tj][tk];
        s = s - Qc[c];
        // Res = Fc - Fv - Fd with Fv = Fd = 0 for the inviscid upwind path
        B.R[c * box + x] = (s - 0.0) - 0.0;
    }
    if (store_faces) {
        for (int c = 0; c < 5; ++c) {
            fI0[c * box + x] = sI[c][ti][tj][tk];
            fJ0[c * box + x] = sJ[c][ti][tj][tk];
            fK0[c * box + x] = sK[c][ti][tj][tk];
            if (ti == TI - 1 || i == B.ni) fI0[c * box + x + B.si] = sI[c][ti + 1][tj][tk];
            if (tj == TJ - 1 || j == B.nj) fJ0[c * box + x + B.sj] = sJ[c][ti][tj + 1][tk];
            if (tk == TK - 1 || k == B.nk) fK0[c * box + x + 1] = sK[c][ti][tj][tk + 1];
        }
    }
}

#define FV3D_CONV_M(M, A, B, C, NT) \
    template __global__ void k_convective<A, B, C, M, NT>(const BlockDev *, const int4 *, Gas, int, int, double *, double *, \
                                                          double *);
#define FV3D_CONV(S, A, B, C) FV3D_CONV_M(0, A, B, C, 256) FV3D_CONV_M(1, A, B, C, 256) FV3D_CONV_M(2, A, B, C, 256)
FV3D_FOR_TILES(FV3D_CONV)
FV3D_CONV_M(0, 4, 4, 16, conv_wide(0))
FV3D_CONV_M(1, 4, 4, 16, conv_wide(1))
FV3D_CONV_M(2, 4, 4, 16, conv_wide(2))
#undef FV3D_CONV
#undef FV3D_CONV_M

// Face-parallel form of the same residual: every face of every block once, one
// thread per face (faces of a block and direction i-slowest, k fastest), into
// B.fcv; k_conv_sum then forms each cell's residual from its six faces and the
// rotation source in k_convective's order, so the two forms agree bit for bit.
template <int MODE>
__global__ void __launch_bounds__(256) k_conv_faces(const BlockDev *__restrict__ blocks, const long *__restrict__ fstart,
                                                    int nlist, Gas g)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= fstart[nlist]) return;
    const int q = find_range(fstart, nlist, t);
    const int d = q % 3;
    BlockRef B = block_at(blocks, q / 3);
    const long r = t - fstart[q];
    const int nj = B.nj + (d == 1 ? 1 : 0), nk = B.nk + (d == 2 ? 1 : 0);
    const int i = (int)(r / ((long)nj * nk)) + 1, j = (int)(r / nk % nj) + 1, k = (int)(r % nk) + 1;
    double f[5];
    face_flux<MODE>(B, g, d, i, j, k, f);
    const long x = cidx(B, i, j, k);
    for (int c = 0; c < 5; ++c) B.fcv[(long)(d * 5 + c) * B.box + x] = f[c];
}

template __global__ void k_conv_faces<0>(const BlockDev *, const long *, int, Gas);
template __global__ void k_conv_faces<1>(const BlockDev *, const long *, int, Gas);
template __global__ void k_conv_faces<2>(const BlockDev *, const long *, int, Gas);

__global__ void __launch_bounds__(256) k_conv_sum(const BlockDev *__restrict__ blocks, const long *__restrict__ cstart,
                                                  int nblock, int ndec)
{
    if (blockIdx.x == 0) flag_decrement(blocks, ndec);
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int n, i, j, k;
    if (!cell_item(blocks, cstart, nblock, t, n, i, j, k)) return;
    BlockRef B = block_at(blocks, n);
    const long box = B.box, x = cidx(B, i, j, k);
    const double w_rot = B.w_rot;
    const double vol = B.vol[x];
    const double dens = B.W[x], uvel = B.W[box + x], vvel = B.W[2 * box + x];
    double Qc[5] = {0.0, dens * (w_rot * vvel) * vol, F32C(-1.0) * dens * (w_rot * uvel) * vol, 0.0, 0.0};
    for (int c = 0; c < 5; ++c) {
        const double *FI = B.fcv + (long)c * box, *FJ = B.fcv + (long)(5 + c) * box, *FK = B.fcv + (long)(10 + c) * box;
        double s = FI[x + B.si] - FI[x];
        s = s + FJ[x + B.sj];
        s = s - FJ[x];
        s = s + FK[x + 1];
        s = s - FK[x];
        s = s - Qc[c];
        B.R[c * box + x] = (s - 0.0) - 0.0;
    }
}

// ================================================================ LU-SGS
// Flux difference of CTimeDiscr::delt_Fn_up / delt_Fn_down
// (source/LU_SGS_Marching.cpp:293-419) at neighbour cell nb whose faces along
// d are nb (lower) and nb + stride (upper).
__device__ static void delt_fn(BlockRef B, double Gamma, int d, long nb, double df[5])
{
    const long box = B.box;
    const long st = d == 0 ? B.si : d == 1 ? B.sj : 1;
    const long fa = nb + st, fb = nb;   // upper face first, as the reference sums them
    const double *S = B.fS[d], *s = B.fs[d];
    double nx = (S[fa] / s[fa] + S[fb] / s[fb]) / F32C(2.0);
    double ny = (S[box + fa] / s[fa] + S[box + fb] / s[fb]) / F32C(2.0);
    double nz = (S[2 * box + fa] / s[fa] + S[2 * box + fb] / s[fb]) / F32C(2.0);
    double uvel_e = F32C(-1.0) * B.cc[box + nb] * B.w_rot;
    double vvel_e = B.cc[nb] * B.w_rot;
    double o[5], nw[5];
    for (int c = 0; c < 5; ++c) { o[c] = B.Q[c * box + nb]; nw[c] = o[c] + B.dQ[c * box + nb]; }
    double dens = nw[0], uvel = nw[1] / nw[0], vvel = nw[2] / nw[0], wvel = nw[3] / nw[0], E = nw[4] / nw[0];
    double press_new = (Gamma - F32C(1.0)) * dens * (E - F32C(0.5) * (uvel * uvel + vvel * vvel + wvel * wvel));
    double press_old = B.W[4 * box + nb];
    double Vn_old = o[1] / o[0] * nx + o[2] / o[0] * ny + o[3] / o[0] * nz;
    double Vn_new = uvel * nx + vvel * ny + wvel * nz;
    double Vn_e = uvel_e * nx + vvel_e * ny + F32C(0.0) * nz;
    df[0] = nw[0] * (Vn_new - Vn_e) - o[0] * (Vn_old - Vn_e);
    df[1] = (nw[1] * (Vn_new - Vn_e) + press_new * nx) - (o[1] * (Vn_old - Vn_e) + press_old * nx);
    df[2] = (nw[2] * (Vn_new - Vn_e) + press_new * ny) - (o[2] * (Vn_old - Vn_e) + press_old * ny);
    df[3] = (nw[3] * (Vn_new - Vn_e) + press_new * nz) - (o[3] * (Vn_old - Vn_e) + press_old * nz);
    df[4] = ((nw[4] + press_new) * (Vn_new - Vn_e) + press_new * Vn_e) - ((o[4] + press_old) * (Vn_old - Vn_e) + press_old * Vn_e);
}

// One hyperplane i+j+k = plane of every block.  Thread (n, i, j) handles cell
// (i, j, plane-i-j) of block n.  Cells of one plane depend only on cells of the
// previous plane, so the result equals the reference's serial order exactly.
template <bool FORWARD>
__global__ void k_lusgs_plane(const BlockDev *__restrict__ blocks, const long *__restrict__ pstart, int nblock, int step,
                              double relax, Gas g)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= pstart[nblock]) return;
    const int n = find_range(pstart, nblock, t);
    BlockRef B = block_at(blocks, n);
    const long r = t - pstart[n];
    const int i = (int)(r / B.nj) + 1, j = (int)(r % B.nj) + 1;
    const int last = B.IM + B.JM + B.KM - 3;
    const int plane = FORWARD ? 3 + step : last - step;
    if (plane < 3 || plane > last) return;
    const int k = plane - i - j;
    if (k < 1 || k > B.nk) return;
    const long box = B.box, x = cidx(B, i, j, k);
    const double Gamma = g.gamma;
    double alpha = B.alpha[x];   // Vol/dt + relax*sum(lamc) + 2*sum(lamv), from k_spectral_dt
    double A[3][5], V[3][5];
    const long st[3] = {B.si, B.sj, 1};
    const int pos[3] = {i, j, k};
    const int lim[3] = {B.ni, B.nj, B.nk};
    for (int d = 0; d < 3; ++d) {
        bool ok = FORWARD ? pos[d] != 1 : pos[d] != lim[d];
        if (!ok) {
            for (int c = 0; c < 5; ++c) { A[d][c] = 0.0; V[d][c] = 0.0; }
            continue;
        }
        const long nb = FORWARD ? x - st[d] : x + st[d];
        double df[5];
        delt_fn(B, Gamma, d, nb, df);
        const double *s = B.fs[d];
        double sd = F32C(0.5) * (s[nb] + s[nb + st[d]]);
        double rl = relax * B.lamc[d * box + nb];
        // lamv * dQ (lamv = 0 on the inviscid path)
        double lv = B.lamv ? B.lamv[d * box + nb] : 0.0;
        for (int c = 0; c < 5; ++c) {
            double dq = B.dQ[c * box + nb];
            A[d][c] = FORWARD ? (df[c] * sd + dq * rl) * F32C(0.5) : (df[c] * sd - dq * rl) * F32C(0.5);
            V[d][c] = dq * lv;
        }
    }
    for (int c = 0; c < 5; ++c) {
        double s;
        if (FORWARD) {
            s = B.R[c * box + x] * F32C(-1.0) + A[0][c];
            s = s + A[1][c]; s = s + A[2][c];
        } else {
            s = B.dQ[c * box + x] * alpha - A[0][c];
            s = s - A[1][c]; s = s - A[2][c];
        }
        s = s + V[0][c]; s = s + V[1][c]; s = s + V[2][c];
        B.dQ[c * box + x] = s / alpha;
    }
}

template __global__ void k_lusgs_plane<true>(const BlockDev *, const long *, int, int, double, Gas);
template __global__ void k_lusgs_plane<false>(const BlockDev *, const long *, int, int, double, Gas);

// the row-layout sweep in the arithmetic type T
template <class T>
using gcT = const T __attribute__((address_space(1))) *;
template <class T>
using gT = T __attribute__((address_space(1))) *;
#define TC(x) ((T)(x##f))

namespace {
// row-layout sweep, direction waves: per step the neighbour's static data and the
// terms of the flux difference that do not depend on dQ
template <class T>
struct RowPf {
    T q[5], m[5], p, l, lv, ev;        // state, metrics, pressure, lambda_c, lambda_v, nu~
    T of[5], vn_old, cl;               // old-state flux terms
};
template <int N>
struct Int {
    static constexpr int value = N;
};
// The static loads of a step are issued kStaticAhead steps before it and its
// early terms formed one step before it, so a load has kStaticAhead - 1 steps to
// arrive; a wave cycles through kRing row buffers.  Four steps: with three the
// FP64 sweep of a 1.05M-cell channel takes 424 us instead of 326, with five or more
// the idle steps at a tile's ends cost more than the loads still gain.
constexpr int kStaticAhead = 4;
constexpr int kRing = kStaticAhead + 1;
constexpr int kRowS0 = -kStaticAhead;   // first (idle) step of the row-layout sweep loops
// Keeps a value computed where it stands: the compiler may not move it past a
// later barrier.  No instruction.
__device__ inline void pin(double &x) { asm volatile("" : "+v"(x)); }
__device__ inline void pin(float &x) { asm volatile("" : "+v"(x)); }
// 1/x for the FP32 operator: the hardware reciprocal (within 1 ulp), one
// instruction where a correctly rounded division takes about ten; the FP32
// operator only preconditions the FP64 residual, whose fixed point it keeps
__device__ inline float rcp_op(float x) { return __builtin_amdgcn_rcpf(x); }
// the reciprocal a combine wave divides with: DivBy's (FP64), rcp_op's (FP32)
__device__ inline double recip(double x) { return DivBy(x).r; }
__device__ inline float recip(float x) { return rcp_op(x); }
// whether a mailbox word still holds the empty pattern
__device__ inline bool mbox_empty(double x) { return __builtin_bit_cast(unsigned long long, x) == kMboxEmpty; }
__device__ inline bool mbox_empty(float x) { return __builtin_bit_cast(unsigned int, x) == kMboxEmpty32; }
// the mailbox set of a sweep direction
template <class T>
__device__ inline T *mbox_base(BlockRef B, bool fwd) { return (T *)B.mbox[fwd ? 0 : 1]; }
}  // namespace

// ---------------------------------------------------------------------------
// Tile-skewed sweep layout (BlockDev::srow / sdq).
//
// Lane (tj,tk) of row r of tile (J,K) is cell (r+1-tj-tk, J*TJ+tj+1, K*TK+tk+1).
// k_sweep_fill writes whole rows, one wave per row, giving lanes outside the
// block a harmless unit state; it runs at set-up (metrics and those lanes).
// Each iteration k_sweep_pack copies the state of the cells in; the backward
// sweep leaves its dQ in the cell box.
template <class T>
__global__ void __launch_bounds__(256) k_sweep_fill(const BlockDev *__restrict__ blocks, int block, long nrows, int what)
{
    constexpr int TJ = kKbaTJ, TK = kKbaTK;
    BlockRef B = block_at(blocks, block);
    const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= nrows) return;
    const int lane = threadIdx.x & 63, tj = lane / TK, tk = lane % TK;
    const int slot = (int)(row / B.nr), r = (int)(row % B.nr);
    const int J = slot / B.ntk, K = slot % B.ntk;
    const int i = r + 1 - tj - tk, j = J * TJ + tj + 1, k = K * TK + tk + 1;
    const bool valid = i >= 1 && i <= B.ni && j <= B.nj && k <= B.nk;
    const long box = B.box, x = valid ? cidx(B, i, j, k) : 0;
    T *dst = (T *)B.srow + row * (kSweepQ * 64) + lane;
    if (what & kGatherState) {
        for (int c = 0; c < 5; ++c) dst[(kSQ_Q + c) * 64] = valid ? B.Q[c * box + x] : (c == 0 ? 1.0 : 0.0);
        dst[kSQ_P * 64] = valid ? B.W[4 * box + x] : 1.0;
        for (int d = 0; d < 3; ++d) dst[(kSQ_LAM + d) * 64] = valid ? B.lamc[d * box + x] : 0.0;
        for (int c = 0; c < 5; ++c) dst[(kSQ_R + c) * 64] = valid ? B.R[c * box + x] : 0.0;
        dst[kSQ_A * 64] = valid ? B.alpha[x] : 1.0;
        for (int d = 0; d < 3; ++d) dst[(kSQ_LV + d) * 64] = (valid && B.lamv) ? B.lamv[d * box + x] : 0.0;
        dst[kSQ_EV * 64] = (valid && B.ev) ? B.ev[x] : 0.0;
        dst[kSQ_REV * 64] = (valid && B.res_ev) ? B.res_ev[x] : 0.0;
        dst[kSQ_A2 * 64] = (valid && B.alpha2) ? B.alpha2[x] : 1.0;
    }
    if (what & kGatherMetrics)
        for (int q = 0; q < 15; ++q) dst[(kSQ_SWG + q) * 64] = valid ? B.swg[q * box + x] : 0.0;
}

namespace {
// Work item of workgroup b in a grid of n.  The hardware hands workgroup b to
// XCD b mod 8, so XCD x runs b = x, x + 8, ...; XCD x takes the x-th run of
// consecutive work items, in the order it runs them.  Neighbouring items share
// cache lines at their edges (a 16-cell run of k starts at any offset within a
// 128 B line), which are then fetched into, and written back from, one L2.
__device__ inline long xcd_item(long b, long n)
{
    const long x = b % 8;
    long start = 0;
    for (long y = 0; y < x; ++y) start += (n - y + 7) / 8;   // items of the XCDs before x
    return start + b / 8;
}
// (tile, chunk) of pack work item wg of a block: k tiles fastest, then
// chunks of i, then j tiles, so consecutive items are neighbours along k (they
// share the cell-box lines at their k edges) and items ntk apart neighbours
// along i (they share the partly written rows at their chunk edges)
__device__ inline void pack_item(BlockRef B, long wg, int nchunk, int &slot, int &i0)
{
    const int K = (int)(wg % B.ntk);
    const long rest = wg / B.ntk;
    i0 = (int)(rest % nchunk) * kPackChunk + 1;
    slot = (int)(rest / nchunk) * B.ntk + K;
}
}  // namespace

// One workgroup per (tile, chunk of kPackChunk i-planes, group of quantities):
// the quantities are split into qsplit groups so that a small grid still
// spreads over the chip.  The chunk's cells are read plane by plane along k
// (coalesced) into LDS, then written out row by row: the rows a chunk touches
// are partly written (the lanes whose cell lies in the chunk), each as one
// contiguous run.  The workgroups after the first npack empty the sweeps'
// mailboxes, kFillWords 16-byte words each (a launch of its own before; having
// the sweeps' readers put the pattern back was tried: it cost the FP32 sweeps
// 10 %, more than this).
template <class T>
__global__ void __launch_bounds__(256) k_sweep_pack(const BlockDev *__restrict__ blocks, const long *__restrict__ gstart,
                                                    int nblock, int nq, int qsplit, unsigned npack,
                                                    uint4 *__restrict__ mbox, long nfill)
{
    constexpr int TJ = kKbaTJ, TK = kKbaTK;
    __shared__ double buf[kPackChunk][64];
    if (blockIdx.x >= npack) {
        const unsigned lo = (unsigned)kMboxEmpty, hi = (unsigned)(kMboxEmpty >> 32);
        const uint4 v = sizeof(T) == 4 ? make_uint4(kMboxEmpty32, kMboxEmpty32, kMboxEmpty32, kMboxEmpty32)
                                       : make_uint4(lo, hi, lo, hi);
        const long w0 = (long)(blockIdx.x - npack) * kFillWords, w1 = min(w0 + kFillWords, nfill);
        for (long w = w0 + threadIdx.x; w < w1; w += 256) mbox[w] = v;
        return;
    }
    // the block of this workgroup: gstart holds the running (tile, chunk) counts
    const long item = xcd_item(blockIdx.x, npack);
    const int qg = (int)(item % qsplit);
    const int block = find_range(gstart, nblock, item / qsplit);
    BlockRef B = block_at(blocks, block);
    const long wg = item / qsplit - gstart[block];
    const int nchunk = (B.ni + kPackChunk - 1) / kPackChunk;
    int slot, i0;
    pack_item(B, wg, nchunk, slot, i0);
    const int J = slot / B.ntk, K = slot % B.ntk;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int tj = lane / TK, tk = lane % TK, j = J * TJ + tj + 1, k = K * TK + tk + 1;
    const bool col = j <= B.nj && k <= B.nk;
    const long box = B.box;
    const int NQ = nq;   // 15; 18 with the lamv rows of Navier-Stokes; 21 with the nu~ rows of Spalart-Allmaras
    // the cell-box array and row quantity of each packed quantity
    for (int qi = qg * NQ / qsplit; qi < (qg + 1) * NQ / qsplit; ++qi) {
        const double *src;
        int rq;
        if (qi < 5) { src = B.Q + qi * box; rq = kSQ_Q + qi; }
        else if (qi == 5) { src = B.W + 4 * box; rq = kSQ_P; }
        else if (qi < 9) { src = B.lamc + (qi - 6) * box; rq = kSQ_LAM + qi - 6; }
        else if (qi < 14) { src = B.R + (qi - 9) * box; rq = kSQ_R + qi - 9; }
        else if (qi == 14) { src = B.alpha; rq = kSQ_A; }
        else if (qi < 18) { src = B.lamv + (qi - 15) * box; rq = kSQ_LV + qi - 15; }
        else if (qi == 18) { src = B.ev; rq = kSQ_EV; }
        else if (qi == 19) { src = B.res_ev; rq = kSQ_REV; }
        else { src = B.alpha2; rq = kSQ_A2; }
        for (int ci = w; ci < kPackChunk; ci += 4) {
            const int i = i0 + ci;
            if (col && i <= B.ni) buf[ci][lane] = src[cidx(B, i, j, k)];
        }
        __syncthreads();
        // rows r = i + tj + tk - 1 for i in the chunk
        for (int rr = w; rr < kPackChunk + TJ + TK - 2; rr += 4) {
            const int r = i0 - 1 + rr, i = r + 1 - tj - tk;
            if (col && i >= i0 && i < i0 + kPackChunk && i <= B.ni)
                ((T *)B.srow)[((long)slot * B.nr + r) * (kSweepQ * 64) + rq * 64 + lane] = (T)buf[i - i0][lane];
        }
        __syncthreads();
    }
}

template __global__ void k_sweep_fill<double>(const BlockDev *, int, long, int);
template __global__ void k_sweep_fill<float>(const BlockDev *, int, long, int);
template __global__ void k_sweep_pack<double>(const BlockDev *, const long *, int, int, int, unsigned, uint4 *, long);
template __global__ void k_sweep_pack<float>(const BlockDev *, const long *, int, int, int, unsigned, uint4 *, long);

// The persistent wavefront form of the sweeps, on the tile-skewed layout.  The
// (j,k) cross-section is cut into 4 x 16 tiles, one workgroup per tile; tiles
// are handed out by a ticket counter in topological order, so a tile waits only
// on tiles already running.  A step (one row of the tile, 64 cells) needs the
// dQ of the step before, so the sweep takes about ni + nj + nk steps in a chain
// and its time is the latency of one step.  Everything that does not depend on
// that dQ is therefore taken off the chain, by giving each wave one role:
//   waves 0, 1, 2 (one neighbour direction each): the flux difference and the
//     off-diagonal terms of the step's 64 cells into LDS; while the combine
//     waves work, the loads of the step kStaticAhead on and the terms of the next
//     step that use the old state only (kept there by an empty asm: left alone,
//     the compiler moves them past the barrier, onto the chain);
//   wave 3 (mailbox): reads the dQ that crosses the tile's two upstream edges,
//     ahead of its step, waits for it (bounded) and leaves it in LDS
//     beside the in-tile dQ, so a direction wave reads both alike;
//   waves 4, 5, 6 (combine): each sums two of the components into dQ, keeps dQ in
//     LDS for the next step and stores it (backward: in a ring of the last
//     steps); the right-hand side, the diagonal and its reciprocal are ready
//     before the terms are;
//   wave 7 (store, backward only): dQ back to the cell box.  A plane i of the tile
//     is spread over nineteen steps; when the last of them is in the ring the plane
//     goes out as runs of sixteen cells.  It takes the place of a launch that
//     read the dQ rows back and wrote the box: backward sweep and that launch of the 1.05M-cell
//     channel 320 -> 306 us (FP64), of 2.54M cells 325 -> 314 us (FP32).  The
//     combine waves writing their 64 cells' lines themselves: 441 us.
// Two barriers a step: the terms are in LDS, dQ is in LDS.  With three direction
// waves and one combine wave, each doing its own loads and waits, a step took
// 1.03 us (FP64) and 0.58 us (FP32); it takes 0.58 and 0.40 us.  Forward sweep: 96x32x32
// channel 188 -> 115 us (FP64), 127 -> 83 us (FP32); 1.05M-cell channel 511 -> 323 and
// 348 -> 220 us; 2.54M-cell five-block passage with nu~ 735 -> 435 and 398 -> 275 us.
// Every load is issued unconditionally with clamped indices, so the compiler's
// memory-counter waits are exact.  The per-hyperplane kernel k_lusgs_plane above is the reference's own
// schedule and gives the same bits.
//
// Across a tile edge dQ travels through the upstream tile's mailbox: its
// combine waves store the dQ of its edge lanes there as soon as they have them;
// a word that still holds the empty pattern has not been written (k_sweep_pack
// empties them).  Tiles
// start in ticket order, so every upstream tile is already running.
//
// With SA the nu~ equation of Spalart-Allmaras rides along as a sixth
// component (source/LU_SGS_Marching.cpp:88-157, 178-257): the direction waves
// form (nu~ + dnu~) Vn_new - nu~ Vn_old of their neighbour from the same Vn
// as the flow terms, and the combine wave divides by alpha2.  The reference
// updates both per cell from the same neighbour increments, so this is its
// order.
template <bool FWD, int TJ, int TK, bool VISC, bool SA, class T>
__global__ void __launch_bounds__(sl_threads(FWD)) k_lusgs_sl(const BlockDev *__restrict__ blocks, const KbaTile *__restrict__ tiles,
                                                         int ntiles, int *__restrict__ ticket,
                                                         int *__restrict__ next_ticket, int *__restrict__ err,
                                                         double relax, Gas g)
{
    static_assert(TJ * TK == 64, "64 cells per tile");
    static_assert(!SA || VISC, "Spalart-Allmaras runs with the viscous terms");
    // The FP32 operator forms the flux difference without cancellation; the
    // FP64 one follows the reference's expression order.
    constexpr bool kDeltaForm = sizeof(T) == 4;
    constexpr int NC = SA ? 6 : 5;        // increments carried per cell
    constexpr int kE = 64 + TK + TJ;      // dQ per component: the tile's cells, then the j-edge and k-edge words
    // LDS words are laid out so that a lane moves 16 bytes at a time.
    // dQ of a step, two buffers: FP32 (0..3) of a lane together, FP64 (0,1) and
    // (2,3) in a plane each; then 4 (and nu~).
    constexpr int NR = NC - 4;
    constexpr bool kWide = sizeof(T) == 4;
    __shared__ __align__(16) T sdq[2][kE * 4 + kE * NR];
    auto dqi = [](int c, int l) {
        return c >= 4 ? kE * 4 + l * NR + c - 4 : kWide ? l * 4 + c : (c >> 1) * kE * 2 + l * 2 + (c & 1);
    };
    // off-diagonal terms A and V of components (2p, 2p+1), per direction
    typedef T Pair __attribute__((ext_vector_type(2)));
    typedef T Quad __attribute__((ext_vector_type(4)));
    __shared__ Pair sA[kWide && VISC ? 1 : 3][3][64];
    __shared__ Pair sV[!kWide && VISC ? 3 : 1][3][64];
    __shared__ Quad sAV[kWide && VISC ? 3 : 1][3][64];
    // the final dQ of the last steps, from which the store wave takes planes
    constexpr int kStore = TJ + TK;   // a plane's cells spread over kStore - 1 steps
    __shared__ T ring[FWD ? 1 : kStore][NC][64];
    __shared__ int s_q;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int tj = lane / TK, tk = lane % TK;
    const T Gamma = (T)g.gamma;
    constexpr int RQ = kSweepQ * 64, RD = kSweepD * 64;   // words per row
    // the other direction's tickets, whose sweep runs next
    if (blockIdx.x == 0 && threadIdx.x == 0) *next_ticket = 0;
    for (;;) {
        if (threadIdx.x == 0) s_q = atomicAdd(ticket, 1);
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(s_q);
        __syncthreads();
        if (q >= ntiles) return;
        const KbaTile tl = tiles[q];
        BlockRef B = block_at(blocks, tl.block);
        const int ni = B.ni, nj = B.nj, nk = B.nk, nr = B.nr, ntk = B.ntk;
        const int slot = (tl.j0 / TJ) * ntk + tl.k0 / TK;
        const gcT<T> rows = (gcT<T>)((const T *)B.srow + (long)slot * nr * RQ);
        const gT<T> drows = (gT<T>)((T *)B.sdq + (long)slot * nr * RD);
        const int lj = FWD ? tj : TJ - 1 - tj, lk = FWD ? tk : TK - 1 - tk;
        const int j = tl.j0 + tj + 1, k = tl.k0 + tk + 1;
        const bool col = j <= nj && k <= nk;
        // steps run: [kRowS0, send), a whole number of kRing-step unrollings
        const int send = (nr - kRowS0 + kRing - 1) / kRing * kRing + kRowS0;
        auto clampr = [&](int r) { return min(max(r, 0), nr - 1); };
        // own row of a step.  At step s a lane's cell has l2 = s - lj - lk cells
        // of its column done before it, and exists when 0 <= l2 < ni.
        auto row_of = [&](int step) { return FWD ? step : nr - 1 - step; };
        auto bar = []() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        };
        auto dir_loop = [&](auto dc) {
            constexpr int d = decltype(dc)::value;
            constexpr int TE = d == 1 ? TJ : TK;   // tile extent along d
            const int dep = d == 1 ? tl.dep_j : d == 2 ? tl.dep_k : -1;
            const bool edge = d == 1 ? tj == (FWD ? 0 : TJ - 1) : d == 2 ? tk == (FWD ? 0 : TK - 1) : false;
            const bool from_up = d != 0 && edge && dep >= 0;
            // upstream tile, and its lane facing this lane across the tile edge
            const int uslot = d == 1 ? slot + (FWD ? -ntk : ntk) : slot + (FWD ? -1 : 1);
            const int ulane = d == 1 ? (FWD ? (TJ - 1) * TK : 0) + tk : tj * TK + (FWD ? TK - 1 : 0);
            // in-tile neighbour lane
            const int nlane = (d == 0 || edge) ? lane : d == 1 ? lane + (FWD ? -TK : TK) : lane + (FWD ? -1 : 1);
            // where the neighbour's dQ lies in sdq, and its static row: the lane's
            // column in the row before, or (edge lanes) the upstream tile's row
            const int qlane = (d == 0 || !edge) ? nlane : d == 1 ? 64 + tk : 64 + TK + tj;
            const gcT<T> src0 = from_up ? (gcT<T>)((const T *)B.srow + (long)uslot * nr * RQ) + ulane : rows + nlane;
            const int radd = from_up ? (FWD ? TE - 1 : 1 - TE) : (FWD ? -1 : 1);
            // the lane's neighbour takes part in steps 0 <= s - first < count
            const bool okd = col && (d == 1 ? j != (FWD ? 1 : nj) : d == 2 ? k != (FWD ? 1 : nk) : true);
            const int first = lj + lk + (d == 0 ? 1 : 0), count = okd ? ni - (d == 0 ? 1 : 0) : 0;
            // the neighbour's state and metrics of a step (static during the sweep)
            auto issue_static = [&](RowPf<T> &bn, int step) {
                const gcT<T> src = src0 + (long)clampr(row_of(step) + radd) * RQ;
                for (int c = 0; c < 5; ++c) bn.q[c] = src[(kSQ_Q + c) * 64];
                bn.p = src[kSQ_P * 64];
                bn.l = src[(kSQ_LAM + d) * 64];
                if (VISC) bn.lv = src[(kSQ_LV + d) * 64];
                for (int c = 0; c < 5; ++c) bn.m[c] = src[(kSQ_SWG + d * 5 + c) * 64];
                if constexpr (SA) bn.ev = src[kSQ_EV * 64];
            };
            // the terms of the flux difference that use only the old state
            // (source/LU_SGS_Marching.cpp:293-419; same operations, evaluated early)
            auto precompute = [&](RowPf<T> &b) {
                const T *o = b.q;
                const T nx = b.m[0], ny = b.m[1], nz = b.m[2], Vn_e = b.m[4];
                const T press_old = b.p;
                if constexpr (kDeltaForm) {
                    // old velocity and total enthalpy per volume for the
                    // cancellation-free difference below (one reciprocal of
                    // the density: this operator only preconditions)
                    const T r0 = rcp_op(o[0]);
                    b.of[0] = o[1] * r0;
                    b.of[1] = o[2] * r0;
                    b.of[2] = o[3] * r0;
                    b.of[3] = o[4] + press_old;
                    b.vn_old = b.of[0] * nx + b.of[1] * ny + b.of[2] * nz;
                    pin(b.of[0]); pin(b.of[1]); pin(b.of[2]); pin(b.of[3]);
                } else {
                    const DivBy by(o[0]);
                    const T Vn_old = by.of(o[1]) * nx + by.of(o[2]) * ny + by.of(o[3]) * nz;
                    b.vn_old = Vn_old;
                    b.of[0] = o[0] * (Vn_old - Vn_e);
                    b.of[1] = o[1] * (Vn_old - Vn_e) + press_old * nx;
                    b.of[2] = o[2] * (Vn_old - Vn_e) + press_old * ny;
                    b.of[3] = o[3] * (Vn_old - Vn_e) + press_old * nz;
                    b.of[4] = (o[4] + press_old) * (Vn_old - Vn_e) + press_old * Vn_e;
                    for (int c = 0; c < 5; ++c) pin(b.of[c]);
                }
                b.cl = (T)relax * b.l;
                pin(b.cl);
                pin(b.vn_old);
            };
            // step s: the dQ-dependent part of the flux difference, the step's terms
            auto chain = [&](const RowPf<T> &b, int s) {
                const bool use = (unsigned)(s - first) < (unsigned)count;
                T dqn[NC];
                {
                    const T *from = sdq[(s - 1) & 1];
                    if constexpr (kWide) {
                        const Quad v = *(const Quad *)(from + dqi(0, qlane));
                        for (int c = 0; c < 4; ++c) dqn[c] = v[c];
                    } else {
                        const Pair v = *(const Pair *)(from + dqi(0, qlane)), w = *(const Pair *)(from + dqi(2, qlane));
                        dqn[0] = v[0]; dqn[1] = v[1]; dqn[2] = w[0]; dqn[3] = w[1];
                    }
                    for (int c = 4; c < NC; ++c) dqn[c] = from[dqi(c, qlane)];
                }
                const T nx = b.m[0], ny = b.m[1], nz = b.m[2], sd = b.m[3], Vn_e = b.m[4];
                T df[5];
                T vn_new = T(0), dvn = T(0);   // the neighbour's new normal velocity and its change
                if constexpr (kDeltaForm) {
                    // F_n(Q+dQ) - F_n(Q) written as sums of products with a
                    // difference factor, so its rounding error scales with dQ:
                    //   du = (dm - u d rho)/(rho + d rho),  dVn = du.n,
                    //   dp = (gamma-1)(dE - (m.du + dm.u')/2),  w' = Vn' - Vn_e
                    //   d(rho w) = d rho w' + rho dVn,  d(m w + p n) = dm w' + m dVn + dp n,
                    //   d((E+p) w + p Vn_e) = (dE + dp) w' + (E+p) dVn + dp Vn_e
                    const T *q = b.q;
                    const T r1 = rcp_op(q[0] + dqn[0]);
                    const T du = (dqn[1] - b.of[0] * dqn[0]) * r1, dv = (dqn[2] - b.of[1] * dqn[0]) * r1,
                            dw = (dqn[3] - b.of[2] * dqn[0]) * r1;
                    const T u1 = b.of[0] + du, v1 = b.of[1] + dv, w1 = b.of[2] + dw;
                    const T dVn = du * nx + dv * ny + dw * nz;
                    const T wn = (b.vn_old + dVn) - Vn_e;
                    const T dp = (Gamma - TC(1.0)) *
                                 (dqn[4] - TC(0.5) * ((q[1] * du + q[2] * dv + q[3] * dw) +
                                                      (dqn[1] * u1 + dqn[2] * v1 + dqn[3] * w1)));
                    vn_new = b.vn_old + dVn;
                    dvn = dVn;
                    df[0] = dqn[0] * wn + q[0] * dVn;
                    df[1] = dqn[1] * wn + q[1] * dVn + dp * nx;
                    df[2] = dqn[2] * wn + q[2] * dVn + dp * ny;
                    df[3] = dqn[3] * wn + q[3] * dVn + dp * nz;
                    df[4] = (dqn[4] + dp) * wn + b.of[3] * dVn + dp * Vn_e;
                } else {
                    T nw[5];
                    for (int c = 0; c < 5; ++c) nw[c] = b.q[c] + dqn[c];
                    const DivBy by(nw[0]);
                    T dens = nw[0], uvel = by.of(nw[1]), vvel = by.of(nw[2]), wvel = by.of(nw[3]), E = by.of(nw[4]);
                    T press_new = (Gamma - TC(1.0)) * dens * (E - TC(0.5) * (uvel * uvel + vvel * vvel + wvel * wvel));
                    T Vn_new = uvel * nx + vvel * ny + wvel * nz;
                    vn_new = Vn_new;
                    df[0] = nw[0] * (Vn_new - Vn_e) - b.of[0];
                    df[1] = (nw[1] * (Vn_new - Vn_e) + press_new * nx) - b.of[1];
                    df[2] = (nw[2] * (Vn_new - Vn_e) + press_new * ny) - b.of[2];
                    df[3] = (nw[3] * (Vn_new - Vn_e) + press_new * nz) - b.of[3];
                    df[4] = ((nw[4] + press_new) * (Vn_new - Vn_e) + press_new * Vn_e) - b.of[4];
                }
                T A[6] = {}, V[6] = {};
                for (int c = 0; c < 5; ++c) {
                    A[c] = FWD ? (df[c] * sd + dqn[c] * b.cl) * TC(0.5) : (df[c] * sd - dqn[c] * b.cl) * TC(0.5);
                    if (VISC) V[c] = dqn[c] * b.lv;   // lamv * dQ
                }
                if constexpr (SA) {
                    // (nu~ + dnu~) Vn_new - nu~ Vn_old (source/LU_SGS_Marching.cpp:351-353); the
                    // FP32 operator writes it as nu~ dVn + dnu~ Vn_new
                    const T dev = dqn[5];
                    T dfe;
                    if constexpr (kDeltaForm) {
                        dfe = b.ev * dvn + dev * vn_new;
                    } else {
                        (void)dvn;
                        const T ev_new = b.ev + dev;
                        dfe = ev_new * vn_new - b.ev * b.vn_old;
                    }
                    A[5] = FWD ? (dfe * sd + b.cl * dev) * TC(0.5) : (dfe * sd - b.cl * dev) * TC(0.5);
                    V[5] = b.lv * dev;
                }
                // a lane without this neighbour contributes zero (few steps have any)
                if (__builtin_amdgcn_ballot_w64(!use))
                    for (int c = 0; c < NC; ++c) {
                        A[c] = use ? A[c] : T(0);
                        if (VISC) V[c] = use ? V[c] : T(0);
                    }
                for (int p = 0; p < 3; ++p) {
                    if constexpr (kWide && VISC) sAV[d][p][lane] = Quad{A[2 * p], A[2 * p + 1], V[2 * p], V[2 * p + 1]};
                    else sA[d][p][lane] = Pair{A[2 * p], A[2 * p + 1]};
                    if constexpr (!kWide && VISC) sV[d][p][lane] = Pair{V[2 * p], V[2 * p + 1]};
                }
            };
            // The loop starts kStaticAhead idle steps early (every lane idle) so
            // that no load precedes it and every step runs the same code;
            // nothing is in flight on entry.
            // b[u] serves step s0 + u: its static data are issued kStaticAhead steps
            // ahead, into the buffer the previous step has finished with
            RowPf<T> b[kRing] = {};
            __builtin_amdgcn_s_waitcnt(0);
            for (int s0 = kRowS0; s0 < send; s0 += kRing) {
#pragma unroll
                for (int u = 0; u < kRing; ++u) {
                    chain(b[u], s0 + u);
                    bar();   // terms of the step are in LDS
                    issue_static(b[(u + kStaticAhead) % kRing], s0 + u + kStaticAhead);
                    precompute(b[(u + 1) % kRing]);
                    bar();   // dQ of the step is in LDS
                }
            }
        };
        // ---- mailbox wave: the upstream dQ of step s + 1 into the buffer that
        // holds the dQ of step s
        auto mail_loop = [&]() {
            constexpr int NJ = TK * NC, NW = (TK + TJ) * NC;   // words: the j edge's, then the k edge's
            gT<T> src[2];
            int radd[2], first[2], count[2], dst[2];
            for (int h = 0; h < 2; ++h) {
                const int w = lane + 64 * h;
                const bool onj = w < NJ;
                const int v = onj ? w : w - NJ, c = onj ? v / TK : v / TJ, e = onj ? v % TK : v % TJ;
                // the edge cell that needs the word
                const int ej = onj ? (FWD ? 0 : TJ - 1) : e, ek = onj ? e : (FWD ? 0 : TK - 1);
                const bool ok = w < NW && (onj ? tl.dep_j : tl.dep_k) >= 0 && tl.j0 + ej < nj && tl.k0 + ek < nk;
                const int uslot = !ok ? slot : onj ? slot + (FWD ? -ntk : ntk) : slot + (FWD ? -1 : 1);
                src[h] = (gT<T>)(mbox_base<T>(B, FWD) + (long)uslot * nr * kMboxRow) + (!ok ? 0 : onj ? v : kMboxJ + v);
                radd[h] = FWD ? (onj ? TJ : TK) - 1 : 1 - (onj ? TJ : TK);
                first[h] = (FWD ? ej : TJ - 1 - ej) + (FWD ? ek : TK - 1 - ek);
                count[h] = ok ? ni : 0;
                dst[h] = w < NW ? dqi(c, 64 + (onj ? e : TK + e)) : -1;
            }
            auto poll = [&](T x[2], int s) {
                for (int h = 0; h < 2; ++h)
                    x[h] = __hip_atomic_load(src[h] + (long)clampr(row_of(s) + radd[h]) * kMboxRow, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
            };
            auto missing = [&](const T x[2], int s) {
                bool m = false;
                for (int h = 0; h < 2; ++h) m = m || ((unsigned)(s - first[h]) < (unsigned)count[h] && mbox_empty(x[h]));
                return __builtin_amdgcn_ballot_w64(m) != 0;
            };
            // Row s + 1 is read as step s - 1 starts and goes to LDS as step s
            // starts.  A read takes about as long as a step and its rest overlaps
            // the direction waves; reading a step earlier keeps the tile a step
            // further behind its neighbour, over some thirty tiles in a row, and
            // reading later (between the barriers) holds up every step.
            // Measured, forward sweep, FP64 / FP32: 1.05M-cell channel 321 / 248 us
            // as here, 335 / 220 a step earlier, 410 / 305 later; 96x32x32 channel
            // 111 / 82, 120 / 86, 112 / 87.  (All with FP32 rows of FP64 length; at
            // half of it, as now, the 1.05M cells take 220 us as here.)
            T x[2] = {};
            __builtin_amdgcn_s_waitcnt(0);
            for (int s = kRowS0; s < send; ++s) {
                // bounded wait: a run-out sets the error word
                long spins = 0;
                while (missing(x, s + 1)) {
                    poll(x, s + 1);
                    if (++spins > (1L << 22)) { if (lane == 0) atomicExch(err, 1); break; }
                }
                T *to = sdq[s & 1];
                for (int h = 0; h < 2; ++h)
                    if (dst[h] >= 0) to[dst[h]] = x[h];
                poll(x, s + 2);
                bar();
                bar();
            }
        };
        // ---- combine waves (source/LU_SGS_Marching.cpp:155, 255): wave p takes the
        // components 2p and 2p + 1
        auto combine_loop = [&](auto pc) {
            constexpr int p = decltype(pc)::value, C0 = 2 * p, N = NC - C0 < 2 ? NC - C0 : 2;
            constexpr bool kNu = C0 + N > 5;   // with the nu~ one
            const gT<T> mbox = (gT<T>)(mbox_base<T>(B, FWD) + (long)slot * nr * kMboxRow);
            // downstream edges of this tile: the j edge (lanes tj = jl, word tk)
            // and the k edge (lanes tk = kl, word tj)
            const bool jedge = tj == (FWD ? TJ - 1 : 0), kedge = tk == (FWD ? TK - 1 : 0);
            const int count = col ? ni : 0;
            struct Rhs {
                T r[2], a[2];   // right-hand side (backward: the forward dQ) and diagonal per component
                T ra[2];        // reciprocals of the diagonals
            };
            auto issue = [&](Rhs &b, int step) {
                const int ro = clampr(row_of(step));
                const gcT<T> row = rows + (long)ro * RQ + lane, drow = (gcT<T>)drows + (long)ro * RD + lane;
                for (int c = 0; c < N; ++c)
                    b.r[c] = !FWD ? drow[(C0 + c) * 64] : C0 + c < 5 ? row[(kSQ_R + C0 + c) * 64] : row[kSQ_REV * 64];
                b.a[0] = row[kSQ_A * 64];
                if (kNu) b.a[1] = row[kSQ_A2 * 64];
            };
            // what does not depend on the step's terms
            auto prepare = [&](Rhs &b) {
                if (!kNu) b.a[1] = b.a[0];
                b.ra[0] = recip(b.a[0]);
                pin(b.ra[0]);
                b.ra[1] = b.ra[0];
                if (kNu) { b.ra[1] = recip(b.a[1]); pin(b.ra[1]); }
                for (int c = 0; c < N; ++c) {
                    b.r[c] = FWD ? b.r[c] * TC(-1.0) : b.r[c] * b.a[c];
                    pin(b.r[c]);
                }
            };
            Rhs b[kRing] = {};
            int slot_now = 0;   // of the step in the ring
            __builtin_amdgcn_s_waitcnt(0);
            for (int s0 = kRowS0; s0 < send; s0 += kRing) {
#pragma unroll
                for (int u = 0; u < kRing; ++u) {
                    const int s = s0 + u;
                    issue(b[(u + kStaticAhead) % kRing], s + kStaticAhead);
                    prepare(b[u]);
                    const bool valid = (unsigned)(s - lj - lk) < (unsigned)count;
                    bar();
                    Pair A[3], V[3];
                    for (int d = 0; d < 3; ++d) {
                        if constexpr (kWide && VISC) {
                            const Quad v = sAV[d][p][lane];
                            A[d] = Pair{v[0], v[1]};
                            V[d] = Pair{v[2], v[3]};
                        } else {
                            A[d] = sA[d][p][lane];
                            if constexpr (VISC) V[d] = sV[d][p][lane];
                        }
                    }
                    T out[2];
                    for (int c = 0; c < N; ++c) {
                        T v = FWD ? b[u].r[c] + A[0][c] : b[u].r[c] - A[0][c];
                        v = FWD ? v + A[1][c] : v - A[1][c];
                        v = FWD ? v + A[2][c] : v - A[2][c];
                        if constexpr (VISC) { v = v + V[0][c]; v = v + V[1][c]; v = v + V[2][c]; }
                        if constexpr (kDeltaForm) out[c] = v * b[u].ra[c];
                        else out[c] = DivBy(b[u].a[c], b[u].ra[c]).of(v);
                    }
                    if (valid) {
                        T *to = sdq[s & 1] + dqi(C0, lane);
                        if constexpr (N == 2) *(Pair *)to = Pair{out[0], out[1]};
                        else *to = out[0];
                    }
                    bar();
                    if (valid) {
                        // hand the edge values to the downstream tiles, then keep dQ
                        const int ro = row_of(s);
                        const gT<T> mb = mbox + (long)ro * kMboxRow;
                        if (jedge)
                            for (int c = 0; c < N; ++c)
                                __hip_atomic_store(mb + tk + (C0 + c) * TK, out[c], __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
                        if (kedge)
                            for (int c = 0; c < N; ++c)
                                __hip_atomic_store(mb + kMboxJ + tj + (C0 + c) * TJ, out[c], __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
                        for (int c = 0; c < N; ++c) {
                            if constexpr (FWD) drows[(long)ro * RD + (C0 + c) * 64 + lane] = out[c];
                            else ring[slot_now][C0 + c][lane] = out[c];
                        }
                    }
                    slot_now = slot_now == kStore - 1 ? 0 : slot_now + 1;
                }
            }
        };
        // ---- store wave (backward): the cells of plane i, each from the step that
        // formed it, into the cell box, once the last of them is in the ring
        auto store_loop = [&]() {
            double *const dst = B.dQ + cidx(B, 0, j, k);
            int sl = lj + lk + 1;   // ring slot of this lane's cell of the plane
            T v[NC];
            auto fetch = [&]() {
                for (int c = 0; c < NC; ++c) v[c] = ring[sl][c][lane];
                sl = sl == kStore - 1 ? 0 : sl + 1;
            };
            auto put = [&](int s) {
                const int i = ni + kStore - 1 - s;
                if (col && i >= 1 && i <= ni) {
                    const long x = (long)i * B.si;
                    for (int c = 0; c < 5; ++c) dst[c * B.box + x] = (double)v[c];
                    if constexpr (SA) B.dev[cidx(B, 0, j, k) + x] = (double)v[5];
                }
            };
            // the stores go out beside the direction waves, the longer half of a step
            for (int s = kRowS0; s < send; ++s) {
                bar();
                fetch();
                bar();
                put(s);
            }
            bar();
            fetch();
            put(send);
        };
        if (wave == 0) dir_loop(Int<0>());
        else if (wave == 1) dir_loop(Int<1>());
        else if (wave == 2) dir_loop(Int<2>());
        else if (wave == 3) mail_loop();
        else if (wave == 4) combine_loop(Int<0>());
        else if (wave == 5) combine_loop(Int<1>());
        else if (wave == 6) combine_loop(Int<2>());
        else if constexpr (!FWD) store_loop();
        if constexpr (!FWD)
            if (wave < 7) bar();   // the store wave's last plane
    }
}

#define FV3D_SL(F, V, S, T) \
    template __global__ void k_lusgs_sl<F, kKbaTJ, kKbaTK, V, S, T>(const BlockDev *, const KbaTile *, int, int *, int *, int *, double, Gas);
FV3D_SL(true, false, false, double)
FV3D_SL(false, false, false, double)
FV3D_SL(true, true, false, double)
FV3D_SL(false, true, false, double)
FV3D_SL(true, true, true, double)
FV3D_SL(false, true, true, double)
FV3D_SL(true, false, false, float)
FV3D_SL(false, false, false, float)
FV3D_SL(true, true, false, float)
FV3D_SL(false, true, false, float)
FV3D_SL(true, true, true, float)
FV3D_SL(false, true, true, float)
#undef FV3D_SL

__global__ void k_fill_u64(unsigned long long *p, long n, unsigned long long v)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

__global__ void k_fill_i32(int *p, int n, int v)
{
    for (int e = threadIdx.x; e < n; e += blockDim.x) p[e] = v;
}

__global__ void k_fill_int(int *p, long n, int v)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

// The values of cells t0 .. t0 + n - 1 of a field, C components each, together
// per cell: cell t is (i, j, k) of an n1 x n2 x n3 box whose first cell has
// indices lo, k fastest.  Interleaved here, a field goes to the caller in
// one copy: 2.54M cells of cv take 12 ms, most of it the copy into fresh host
// pages; interleaving them on the host took 31.
__global__ void __launch_bounds__(256) k_field_rows(const double *__restrict__ src, long box, int C, int si, int sj, int lo,
                                                    int n2, int n3, long t0, long n, double *__restrict__ out)
{
    const long r = (long)blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    const long t = t0 + r;
    const int k = (int)(t % n3), j = (int)(t / n3 % n2);
    const long i = t / n3 / n2, x = (i + lo) * si + (long)(j + lo) * sj + k + lo;
    for (int c = 0; c < C; ++c) out[r * C + c] = src[c * box + x];
}

// ===================================================== update + norms
// Q += dQ (source/LU_SGS_Marching.cpp:262-287), Res_Calculate terms
// (source/ComputeAllBlockVars.cpp:340-357), PrimitiveVars
// (source/PrimitiveVars.cpp:7-29) and the Limit_Vars trigger test
// (source/Limit_FlowVars.cpp:28-29).  One partial sum per workgroup.  With
// Spalart-Allmaras (sa set) also nu~ += dnu~ (source/LU_SGS_Marching.cpp:271-272)
// and, when sa_hi is given, the flag of a block holding a value the limiter
// replaces by its neighbours' mean (above 1000).
__global__ void __launch_bounds__(256) k_update(const BlockDev *__restrict__ blocks, const long *__restrict__ cstart, int nblock,
                                                Gas g, double *__restrict__ partial, int *__restrict__ bad_flag,
                                                int *__restrict__ sa_hi, int sa)
{
    __shared__ double red[5][256];
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double rm[5] = {0, 0, 0, 0, 0};
    for_cell_item(blocks, cstart, nblock, t, [&](BlockRef B, int n, int i, int j, int k) {
        const long box = B.box, x = cidx(B, i, j, k);
        double q[5];
        const double vol = B.vol[x];
        for (int c = 0; c < 5; ++c) {
            double o = B.Q[c * box + x];
            q[c] = o + B.dQ[c * box + x];
            rm[c] = fabs((o - q[c]) / o) * vol;
            B.Q[c * box + x] = q[c];
        }
        const double Gamma = g.gamma, Rgas = g.rgas;
        double d = q[0], u = q[1] / q[0], v = q[2] / q[0], w = q[3] / q[0];
        double V2 = u * u + v * v + w * w;
        double p = (Gamma - F32C(1.0)) * (q[4] - q[0] * V2 / F32C(2.0));
        double T = p / d / Rgas;
        B.W[x] = d; B.W[box + x] = u; B.W[2 * box + x] = v; B.W[3 * box + x] = w; B.W[4 * box + x] = p; B.W[5 * box + x] = T;
        const double dmin = F32C(1.0E-6), dmax = F32C(1000.0), vmax = F32C(1000.0);
        if (d < dmin || d > dmax || p < dmin || p > dmax || u > vmax || v > vmax || w > vmax) atomicOr(bad_flag + n, 1);
        if (sa) {
            const double e = B.ev[x] + B.dev[x];
            B.ev[x] = e;
            if (sa_hi && e > F32C(1000.0)) atomicOr(sa_hi + n, 1);
        }
    });
    for (int c = 0; c < 5; ++c) red[c][threadIdx.x] = rm[c];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int c = 0; c < 5; ++c) red[c][threadIdx.x] = red[c][threadIdx.x] + red[c][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 5; ++c) partial[(long)c * gridDim.x + blockIdx.x] = red[c][0];
}

// the limiter's test of a cell (source/Limit_FlowVars.cpp:28-29)
__device__ static bool bad_cell(BlockRef B, long x)
{
    const long box = B.box;
    const double dmin = F32C(1.0E-6), dmax = F32C(1000.0), vmax = F32C(1000.0);
    double d = B.W[x], p = B.W[4 * box + x];
    return d < dmin || d > dmax || p < dmin || p > dmax || B.W[box + x] > vmax || B.W[2 * box + x] > vmax ||
           B.W[3 * box + x] > vmax;
}

// Limit_Vars (source/Limit_FlowVars.cpp:8-119) in the reference's serial order:
// cells are repaired one after the other, so later repairs see earlier ones.
//
// Res_Calculate runs after Limit_Vars in the reference
// (source/LU_SGS_Marching.cpp:287-290, source/Solver.cpp:92-93), but k_update
// formed the norm partials from the state before the repair.  With partial
// given, each repaired cell's |(q_old - q)/q_old| Vol terms are moved from the
// pre-repair value to the repaired one in its 256-cell group's partial
// (q_old = the pre-repair value minus dQ).  Without it (the limiter after a
// prolongation, which no norm follows) nothing is patched.
__device__ static void limit_vars(const BlockDev *__restrict__ blocks, int nblock, const Gas &g, int *__restrict__ bad_flag,
                                  const long *__restrict__ cstart, double *__restrict__ partial, int npart)
{
    const double Gamma = g.gamma, Rgas = g.rgas;
    const double dmin = F32C(1.0E-6), dmax = F32C(1000.0), vmax = F32C(1000.0);
    for (int n = 0; n < nblock; ++n) {
        if (!bad_flag[n]) continue;
        bad_flag[n] = 0;
        BlockRef B = block_at(blocks, n);
        const long box = B.box;
        int nneg = 0;
        for (int i = 1; i <= B.ni; ++i)
            for (int j = 1; j <= B.nj; ++j)
                for (int k = 1; k <= B.nk; ++k) {
                    const long x = cidx(B, i, j, k);
                    if (!bad_cell(B, x)) continue;
                    nneg++;
                    int kn = 0, i1 = 0, j1 = 0, k1 = 0;
                    double d = 0.0, u = 0.0, v = 0.0, w = 0.0, p = 0.0;
                    for (int ia = -1; ia <= 1; ++ia)
                        for (int ja = -1; ja <= 1; ++ja)
                            for (int ka = -1; ka <= 1; ++ka) {
                                k1 = k + ka; j1 = j + ja; i1 = i + ia;
                                if (i1 > 0 && i1 < B.IM && j1 > 0 && j1 < B.JM && k1 > 0 && k1 < B.KM) {
                                    const long y = cidx(B, i1, j1, k1);
                                    if (!bad_cell(B, y)) {
                                        d = d + B.W[y]; u = u + B.W[box + y]; v = v + B.W[2 * box + y];
                                        w = w + B.W[3 * box + y]; p = p + B.W[4 * box + y];
                                        kn = kn + 1;
                                    }
                                }
                            }
                    if (kn == 0) {
                        const long y = cidx(B, i1, j1, k1);
                        d = B.W[y]; u = B.W[box + y]; v = B.W[2 * box + y]; w = B.W[3 * box + y]; p = B.W[4 * box + y];
                        if (d < dmin) d = dmin;
                        if (d > dmax) d = dmax;
                        if (p < dmin) p = dmin;
                        if (p > dmax) p = dmax;
                        if (fabs(u) > vmax) u = u < 0 ? -fabs(vmax) : fabs(vmax);
                        if (fabs(v) > vmax) v = v < 0 ? -fabs(vmax) : fabs(vmax);
                        if (fabs(w) > vmax) w = w < 0 ? -fabs(vmax) : fabs(vmax);
                    } else {
                        double sn1 = (double)(1.0f / (float)kn);
                        d = d * sn1; u = u * sn1; v = v * sn1; w = w * sn1; p = p * sn1;
                    }
                    B.W[x] = d; B.W[box + x] = u; B.W[2 * box + x] = v; B.W[3 * box + x] = w; B.W[4 * box + x] = p;
                    B.W[5 * box + x] = p / d / Rgas;
                    double qn[5];
                    qn[0] = d; qn[1] = d * u; qn[2] = d * v; qn[3] = d * w;
                    qn[4] = p / (Gamma - F32C(1.0)) + d * (u * u + v * v + w * w) / F32C(2.0);
                    if (partial) {
                        const long t = cstart[n] + ((long)(i - 1) * B.nj + (j - 1)) * B.nk + (k - 1);
                        const double vol = B.vol[x];
                        for (int c = 0; c < 5; ++c) {
                            const double qp = B.Q[c * box + x], o = qp - B.dQ[c * box + x];
                            partial[(long)c * npart + t / 256] += fabs((o - qn[c]) / o) * vol - fabs((o - qp) / o) * vol;
                        }
                    }
                    for (int c = 0; c < 5; ++c) B.Q[c * box + x] = qn[c];
                }
        if (nneg > 0) *B.flag_low_dt = 10;
    }
}

// CFluidProps::Limit_SA (source/Limit_FlowVars.cpp:122-168).  Raising values
// below 1e-8 is pointwise; replacing a value above 1000 by the mean of its
// admissible neighbours depends on the neighbours' already limited values, so
// a block with such a value (k_update flags it) is limited by one thread in
// the reference's order here, and the floor of the other blocks is applied in
// k_sa_res.
__device__ static void limit_sa(const BlockDev *__restrict__ blocks, int nblock, int *__restrict__ hi_flag)
{
    const double SAmin = F32C(1.0E-8), LSAmax = F32C(1000.0);
    for (int n = 0; n < nblock; ++n) {
        if (!hi_flag[n]) continue;
        hi_flag[n] = 0;
        BlockRef B = block_at(blocks, n);
        const int IM = B.IM, JM = B.JM, KM = B.KM;
        for (int i = 1; i <= B.ni; ++i)
            for (int j = 1; j <= B.nj; ++j)
                for (int k = 1; k <= B.nk; ++k) {
                    double *e = B.ev + cidx(B, i, j, k);
                    if (*e < SAmin) *e = SAmin;
                    if (*e > LSAmax) {
                        double s0 = 0.0;
                        int kn = 0;
                        for (int ka = -1; ka <= 1; ++ka)
                            for (int ja = -1; ja <= 1; ++ja)
                                for (int ia = -1; ia <= 1; ++ia) {
                                    const int k1 = k + ka, j1 = j + ja, i1 = i + ia;
                                    if (i1 > 0 && i1 < IM && j1 > 0 && j1 < JM && k1 > 0 && k1 < KM) {
                                        const double v = B.ev[cidx(B, i1, j1, k1)];
                                        if (v >= SAmin && v <= LSAmax) { s0 = s0 + v; kn = kn + 1; }
                                    }
                                }
                        *e = kn == 0 ? LSAmax : s0 / kn;
                    }
                }
    }
}

// The limiters, when k_update (or the multigrid transfers) flagged a bad cell:
// one wave looks at all the flags at once and returns, its first thread
// repairs.  One thread walking the flags of Limit_Vars, and a second launch for
// those of Limit_SA, cost 4.5 us each; a launch that has nothing to do costs
// that much whatever it looks at.
__global__ void __launch_bounds__(64) k_limiter_serial(const BlockDev *__restrict__ blocks, int nblock, Gas g,
                                                       int *__restrict__ bad_flag, const long *__restrict__ cstart,
                                                       double *__restrict__ partial, int npart, int *__restrict__ sa_hi)
{
    int any = 0;
    for (int n = threadIdx.x; n < nblock; n += 64) any |= bad_flag[n] | (sa_hi ? sa_hi[n] : 0);
    if (__builtin_amdgcn_ballot_w64(any != 0) == 0 || threadIdx.x != 0) return;
    limit_vars(blocks, nblock, g, bad_flag, cstart, partial, npart);
    if (sa_hi) limit_sa(blocks, nblock, sa_hi);
}

// ============================================= section integrals, norms
// Mass flow, mass-averaged total pressure and total temperature over one K
// plane (source/Ouput.cpp:9-95): workgroup `part` of section sec sums the cells
// part*256 + t, (part + kSecParts)*256 + t, ... with a fixed-order tree into
// sums[(sec*kSecParts + part)*3 + {mass, ptm, ttm}].
__device__ static void section_part(const BlockDev *__restrict__ blocks, const int2 *__restrict__ secs, const Gas &g,
                                    double *__restrict__ sums, int sec, int part, double (*red)[256])
{
    const int2 sc = secs[sec];
    BlockRef B = block_at(blocks, sc.x);
    const int K = sc.y;
    const long box = B.box;
    const double Gamma = g.gamma, Rgas = g.rgas;
    double m = 0.0, pt = 0.0, tt = 0.0;
    for (int f = part * blockDim.x + threadIdx.x; f < B.ni * B.nj; f += kSecParts * blockDim.x) {
        int i = f / B.nj + 1, j = f % B.nj + 1;
        long a = cidx(B, i, j, K), z = cidx(B, i, j, K - 1);
        double dens = F32C(0.5) * (B.W[a] + B.W[z]), u = F32C(0.5) * (B.W[box + a] + B.W[box + z]);
        double v = F32C(0.5) * (B.W[2 * box + a] + B.W[2 * box + z]), w = F32C(0.5) * (B.W[3 * box + a] + B.W[3 * box + z]);
        const double *S = B.fS[2];
        double mc = dens * (u * S[a] + v * S[box + a] + w * S[2 * box + a]);
        double temp = F32C(0.5) * (B.W[5 * box + a] + B.W[5 * box + z]);
        double Ma = sqrt(u * u + v * v + w * w) / sqrt(Gamma * Rgas * temp);
        double Pt_cell = B.W[4 * box + a] * pow(F32C(1.0) + (Gamma - F32C(1.0)) / F32C(2.0) * Ma * Ma, Gamma / (Gamma - F32C(1.0)));
        m += mc;
        pt += pow(Pt_cell, (Gamma - F32C(1.0)) / Gamma) * mc;
        tt += B.W[5 * box + a] * (1 + (Gamma - F32C(1.0)) / F32C(2.0) * Ma * Ma) * mc;
    }
    red[0][threadIdx.x] = m; red[1][threadIdx.x] = pt; red[2][threadIdx.x] = tt;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int c = 0; c < 3; ++c) red[c][threadIdx.x] += red[c][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 3; ++c) sums[(sec * kSecParts + part) * 3 + c] = red[c][0];
}

__global__ void __launch_bounds__(256) k_sections(const BlockDev *__restrict__ blocks, const int2 *__restrict__ secs, Gas g,
                                                  double *__restrict__ sums)
{
    __shared__ double red[3][256];
    section_part(blocks, secs, g, sums, blockIdx.x / kSecParts, blockIdx.x % kSecParts, red);
}

// The end of an iteration, 2 nsw + 6 workgroups per instance: nsw per section for
// the integrals' parts, and one per component of the residual norm (the
// fixed-order sum of the update's per-workgroup partials); the instance's last
// workgroup to finish then forms the norms, the performance parameters
// (source/Ouput.cpp:97-107,282-300), the CFL ramp for the next iteration
// (source/Solver.cpp:49-60) and the history row, hist_row or, without it, the
// cursor's next one.  As two launches, the second with one workgroup per
// instance, this took 53 us on a 2.54M-cell passage and 12 on the smallest
// grids, and a copy of the row 4.5 more; now 20 and 8.  A workgroup without
// cells leaves at once: with all 70 counting themselves in, eight passages of one
// batch took 30 us, now 17.
__global__ void __launch_bounds__(256) k_finish(const BlockDev *__restrict__ blocks, const int2 *__restrict__ secs,
                                                const double *__restrict__ partial, int npart,
                                                const int2 *__restrict__ parts, double *__restrict__ secsum,
                                                int *__restrict__ arrived, ScalarsDev *lv, ScalarsDev *ramp, Gas g,
                                                double *__restrict__ hist_row, double *const *__restrict__ cursor,
                                                int ninst, int nsw)
{
    __shared__ double red[3][256];
    __shared__ int s_last;
    const int inst = blockIdx.x / (2 * nsw + 6), part = blockIdx.x % (2 * nsw + 6);
    const int t = threadIdx.x;
    ScalarsDev *sc = lv + inst;
    ramp += inst;
    double *norms = secsum + (long)ninst * 2 * kSecParts * 3 + 6 * inst;
    // component 5: Res_ev of Spalart-Allmaras (k_sa_res)
    const int nc = g.turbulence == 200 ? 6 : 5;
    // section parts that hold cells; the other workgroups have nothing to do
    // (each that counts itself in writes its XCD's L2 back first)
    auto nonempty = [&](int sec) {
        BlockRef B = block_at(blocks, secs[2 * inst + sec].x);
        return min((B.ni * B.nj + 255) / 256, kSecParts);
    };
    const int np0 = nonempty(0), np1 = nonempty(1);
    const int sec = part / nsw, np = sec == 0 ? np0 : np1;
    if (sec < 2 ? part % nsw >= np : part - 2 * nsw >= nc) return;
    if (sec < 2) {
        for (int p = part % nsw; p < np; p += nsw) section_part(blocks, secs, g, secsum, inst * 2 + sec, p, red);
    } else {
        const int c = part - 2 * nsw;
        double r = 0.0;
        // each thread adds partials t, t + 256, ... in that order; sixteen
        // loads are in flight before the first is added
        const double *src = partial + (long)c * npart + parts[inst].x;
        const int n = parts[inst].y;
        int p = t;
        for (; p + 15 * 256 < n; p += 16 * 256) {
            double v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = src[p + u * 256];
#pragma unroll
            for (int u = 0; u < 16; ++u) r += v[u];
        }
        for (; p < n; p += 256) r += src[p];
        red[0][t] = r;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (t < w) red[0][t] += red[0][t + w];
            __syncthreads();
        }
        if (t == 0) norms[c] = red[0][0];
    }
    // what this workgroup wrote (thread 0) is visible before it counts itself in
    if (t == 0) {
        __threadfence();
        s_last = atomicAdd(arrived + inst, 1) == min(np0, nsw) + min(np1, nsw) + nc - 1;
        if (s_last) __threadfence();
    }
    __syncthreads();
    if (!s_last) return;
    const double total_vol = sc->total_vol, dens_ref = sc->dens_ref, vel_ref = sc->vel_ref, temp_ref = sc->temp_ref;
    const double nblade_in = sc->nblade_in, nblade_out = sc->nblade_out;
    // section partials in a fixed order: section 0 inlet, 1 outlet; mass, ptm,
    // ttm; then the norms
    const double *own = secsum + (long)inst * 2 * kSecParts * 3;
    const int e = t / 3;   // part of the partial this thread brings in
    if (t < 2 * kSecParts * 3) {
        if (e % kSecParts < (e < kSecParts ? np0 : np1))
            red[0][t] = __hip_atomic_load(own + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (t < 2 * kSecParts * 3 + 6) {
        const int c = t - 2 * kSecParts * 3;
        red[0][t] = c < nc ? __hip_atomic_load(norms + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
    }
    __syncthreads();
    if (t < 6) {
        double s = 0.0;
        const int m = t < 3 ? np0 : np1;
        for (int p = 0; p < m; ++p) s += red[0][((t / 3) * kSecParts + p) * 3 + t % 3];
        red[1][t] = s;
    }
    __syncthreads();
    const double Gamma = g.gamma, Rgas = g.rgas;
    const double *norm = &red[0][2 * kSecParts * 3], *sums = red[1];
    if (t < 2)
        red[2][t] = pow(sums[3 * t + 1] / sums[3 * t], Gamma / (Gamma - F32C(1.0))) * dens_ref * vel_ref * vel_ref;
    __syncthreads();
    if (t != 0) return;
    arrived[inst] = 0;
    for (int c = 0; c < 5; ++c) sc->res[c] = norm[c] / total_vol;
    sc->res_ev = norm[5] / total_vol;
    double mi = sums[0] * dens_ref * vel_ref * nblade_in;
    double mo = sums[3] * dens_ref * vel_ref * nblade_out;
    const double pti = red[2][0], pto = red[2][1];
    double tti = sums[2] / sums[0] * temp_ref, tto = sums[5] / sums[3] * temp_ref;
    double PR = pto / pti;
    double L_adk = Gamma / (Gamma - F32C(1.0)) * Rgas * tti * (pow(PR, (Gamma - F32C(1.0)) / Gamma) - F32C(1.0));
    double L_k = Gamma / (Gamma - F32C(1.0)) * Rgas * tti * (tto / tti - F32C(1.0));
    ramp->iter += 1;
    if (!hist_row) {
        if (cursor) hist_row = *cursor + 7L * ((long)ramp->hist_pos * ninst + inst);
        ramp->hist_pos += 1;
    } else {
        hist_row += 7L * inst;
    }
    if (hist_row) {
        hist_row[0] = ramp->iter; hist_row[1] = sc->res[0]; hist_row[2] = mi; hist_row[3] = mo;
        hist_row[4] = PR; hist_row[5] = L_adk / L_k; hist_row[6] = ramp->cfl;
    }
    sc->mass_in = mi; sc->mass_out = mo; sc->pr = PR; sc->eff = L_adk / L_k;
    // CFL ramp applied for the next iteration (source/Solver.cpp:49-59), on the
    // density residual of the level that ran
    if (sc->res[0] <= ramp->cfl_res) {
        ramp->cfl = ramp->cfl * F32C(1.2);
        ramp->cfl_res = ramp->cfl_res / F32C(10.0);
    }
    if (ramp->cfl > F32C(10.0)) ramp->cfl = F32C(10.0);
}

// A run of replayed iterations starts: its history goes to hist from row 0.
__global__ void k_hist_begin(double **cursor, double *hist, ScalarsDev *ramp, int ninst)
{
    if (threadIdx.x == 0) *cursor = hist;
    for (int w = threadIdx.x; w < ninst; w += blockDim.x) ramp[w].hist_pos = 0;
}

// ============================================================ mixing plane
// CMesh::BndCondMixingPlane (source/BndCondMixingPlane.cpp:287-522), one
// workgroup per radial line i of a plane.  The threads form the per-face
// terms of each side's pitch-wise sums into LDS; one thread adds them in j
// order (the reference's order) and forms the mixed-out state of each side:
// the flux-averaged mass, momentum, energy (and rho nu~) fluxes, pressure from
// the quadratic of lines 370 / 432, then velocity, density, temperature and
// the speed of sound.  The threads then write the characteristic ghost
// states: block 1's K-high ghosts (and Dummy layers) from the downstream
// average plus its outgoing waves, block 2's K-low ghosts from the upstream
// average plus its outgoing wave; nu~ ghosts take the upstream average.
struct MixAvg {
    double d, u, v, w, p, c, ev;
};

__device__ static void mix_terms(BlockRef B, int i, int j, int kf, int kc, int sa, double *t)
{
    const long xf = cidx(B, i, j, kf), xc = cidx(B, i, j, kc), box = B.box;
    const double s = B.fs[2][xf];
    const double nx = B.fS[2][xf] / s, ny = B.fS[2][box + xf] / s, nz = B.fS[2][2 * box + xf] / s;
    const double u = B.W[box + xc], v = B.W[2 * box + xc], w = B.W[3 * box + xc], p = B.W[4 * box + xc];
    const double Vn = u * nx + v * ny + w * nz;
    t[0] = s;
    t[1] = nx * s;
    t[2] = ny * s;
    t[3] = nz * s;
    t[4] = B.Q[xc] * Vn * s;
    t[5] = (B.Q[box + xc] * Vn + nx * p) * s;
    t[6] = (B.Q[2 * box + xc] * Vn + ny * p) * s;
    t[7] = (B.Q[3 * box + xc] * Vn + nz * p) * s;
    t[8] = (B.Q[4 * box + xc] + p) * Vn * s;
    t[9] = sa ? B.Q[xc] * B.ev[xc] * Vn * s : 0.0;
}

__device__ static MixAvg mix_reduce(const double (*t)[10], int nj, const Gas &g, int sa)
{
    const double Gamma = g.gamma, Rgas = g.rgas;
    double s_sum = 0.0, nsx = 0.0, nsy = 0.0, nsz = 0.0, I[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int j = 0; j < nj; ++j) {
        nsx = nsx + t[j][1];
        nsy = nsy + t[j][2];
        nsz = nsz + t[j][3];
        s_sum = s_sum + t[j][0];
        for (int m = 1; m <= 6; ++m) I[m] = I[m] + t[j][3 + m];
    }
    MixAvg a;
    for (int m = 1; m <= 5; ++m) I[m] = I[m] / s_sum;
    a.ev = 0.0;
    if (sa) {
        I[6] = I[6] / s_sum;
        a.ev = I[6] / I[1];
    }
    const double nx = nsx / s_sum, ny = nsy / s_sum, nz = nsz / s_sum;
    const double tA = I[2] * nx + I[3] * ny + I[4] * nz;
    const double tB = F32C(2.0) * I[1] * I[5] - (I[2] * I[2] + I[3] * I[3] + I[4] * I[4]);
    const double tC = nx * nx + ny * ny + nz * nz;
    a.p = (tA / tC + sqrt(tA * tA / tC / tC - (Gamma * Gamma - F32C(1.0)) * tB / tC)) / (Gamma + F32C(1.0));
    a.u = (I[2] - a.p * nx) / I[1];
    a.v = (I[3] - a.p * ny) / I[1];
    a.w = (I[4] - a.p * nz) / I[1];
    a.d = I[1] / (a.u * nx + a.v * ny + a.w * nz);
    const double T = a.p / Rgas / a.d;
    a.c = sqrt(Gamma * Rgas * T);
    return a;
}

__device__ static void mix_ghost(BlockRef B, int s, int i, int j, int kg, double d, double u, double v,
                                 double w, double p, double ev, const Gas &g, int sa)
{
    const double Gamma = g.gamma, Rgas = g.rgas;
    const double pv[6] = {d, u, v, w, p, p / Rgas / d};
    const double V2 = u * u + v * v + w * w;
    const double cv[5] = {d, d * u, d * v, d * w, p / (Gamma - F32C(1.0)) + d * V2 / F32C(2.0)};
    const long x = cidx(B, i, j, kg), box = B.box;
    for (int c = 0; c < 5; ++c) B.Q[c * box + x] = cv[c];
    for (int c = 0; c < 6; ++c) B.W[c * box + x] = pv[c];
    if (sa) B.ev[x] = ev;
    set_dummies(B, s, i, j, cv, pv);
}

__global__ void __launch_bounds__(256) k_mixing_plane(const BlockDev *__restrict__ blocks,
                                                      const MixDev *__restrict__ mix, int nmix, Gas g, int sa)
{
    __shared__ double t[kMixMaxJ][10];
    __shared__ MixAvg avg[2];
    int q = 0;
    while (q + 1 < nmix && mix[q + 1].line0 <= (int)blockIdx.x) ++q;
    const MixDev M = mix[q];
    const int i = M.i0 + ((int)blockIdx.x - M.line0);
    BlockRef U = block_at(blocks, M.b1), D = block_at(blocks, M.b2);
    const int KM = U.KM;
    for (int side = 0; side < 2; ++side) {
        const int nj = side ? M.nj2 : M.nj1, j0 = side ? M.j2 : M.j1;
        for (int r = threadIdx.x; r < nj; r += blockDim.x)
            mix_terms(side ? D : U, i, j0 + r, side ? 1 : KM, side ? 1 : KM - 1, sa, t[r]);
        __syncthreads();
        if (threadIdx.x == 0) avg[side] = mix_reduce(t, nj, g, sa);
        __syncthreads();
    }
    const MixAvg u = avg[0], d = avg[1];
    for (int r = threadIdx.x; r < M.nj1; r += blockDim.x) {   // lines 460-491
        const int j = M.j1 + r;
        const long x = cidx(U, i, j, KM - 1), box = U.box;
        const double pd = U.W[x], pu = U.W[box + x], pvv = U.W[2 * box + x], pw = U.W[3 * box + x],
                     pp = U.W[4 * box + x];
        const double C1 = -u.c * u.c * (pd - u.d) + (pp - u.p);
        const double C2 = u.d * u.c * (pw - u.w) + (pp - u.p);
        const double C5 = 0.0;
        mix_ghost(U, 5, i, j, KM, d.d + (-C1 + (C2 + C5) / F32C(2.0)) / (d.c * d.c), pu, pvv,
                  d.w + (C2 - C5) / (F32C(2.0) * d.d * d.c), d.p + (C2 + C5) / F32C(2.0), u.ev, g, sa);
    }
    for (int r = threadIdx.x; r < M.nj2; r += blockDim.x) {   // lines 494-522
        const int j = M.j2 + r;
        const long x = cidx(D, i, j, 1), box = D.box;
        const double pw = D.W[3 * box + x], pp = D.W[4 * box + x];
        const double C1 = 0.0, C2 = 0.0, C3 = 0.0, C4 = 0.0;
        const double C5 = (F32C(0.0) - d.d * d.c * (pw - d.w) + (pp - d.p));
        mix_ghost(D, 4, i, j, 0, u.d + (-C1 + (C2 + C5) / F32C(2.0)) / (u.c * u.c), u.u + C4 / (u.d * u.c),
                  u.v + C3 / (u.d * u.c), u.w - C5 / (F32C(2.0) * u.d * u.c), u.p + (C2 + C5) / F32C(2.0), u.ev, g,
                  sa);
    }
}

}  // namespace fv3d
