// shockx.hip -- libshockx.so: gfx950 kernels and the C ABI of the SHOCK RHS / RK-stage path.
//
// Stage pipeline (one RK stage; src/Functions.c:2107-2365):
//   k_ghost_periodic   on-device ghost fill of rho,u,v,w,e along periodic directions (replaces
//                      the MPI self-interface halo, src/Functions.c:3580-3684); all-periodic inviscid
//                      sweeps read ghosts at their image instead
//   k_calc_values      T and mu on every padded node (CalcValues, src/Functions.c:2392-2481;
//                      p, c and theta are recomputed inside the flux kernels instead of stored)
//   k_face_bc          boundary writers of non-periodic faces, in face order (src/BC.c:13-74)
//   k_visc_grad_march  nodal derivatives of u,v,w,T (src/ZD.c:697-810)
//   k_weno             one launch per direction: LDS-staged pencil, characteristic WENO
//                      interface fluxes and their divergence fused, interface fluxes never
//                      reach HBM (CalcFluxesIn*Direction, src/WENO.c:206-1083)
//   k_visc_sweep       one launch per direction: viscous face fluxes and their divergence
//                      (src/ZD.c:47-694); the last one also applies the RK stage update and
//                      the source (src/Functions.c:2287-2365) and writes the next stage state
//                      into another buffer (the reference updates in place after all fluxes of
//                      the stage are assembled, which the separate buffer reproduces exactly)
//   k_weno_last        the last direction's WENO sweep, which applies the update in inviscid runs
//   k_plane            2D: all of the above after the ghost fill in one kernel per stage
// Every hot kernel body is also reachable through a k_*_batch twin that runs many cases from
// one launch over a tile work list (shx_batch_*).
#include "shockx_kernels.h"
#include "../../include/shockx.h"

#include <float.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include <algorithm>
#include <functional>
#include <thread>
#include <vector>

using namespace shx;

// ----------------------------------------------------------------------------------------
// kernels
// ----------------------------------------------------------------------------------------

// Periodic ghost fill of nf fields: every node that is a ghost in a periodic direction copies
// the node at the wrapped index of each periodic direction (fixed point of the ghost-inclusive
// halo passes, src/Functions.c:2117-2136; indices along non-periodic directions are kept, so a
// face slab's ghosts wrap along the periodic tangential directions only).
// node index of the periodic image of padded node idx; ghost: idx is a ghost in a periodic direction
__device__ __forceinline__ long periodic_image(const Geom &gm, const int idx[3], bool &ghost)
{
    ghost = false;
    long src = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        int s = idx[d];
        if (gm.ng[d] > 1 && gm.per[d]) {
            if (s < gm.lo[d]) { s += gm.n[d]; ghost = true; }
            else if (s >= gm.lo[d] + gm.n[d]) { s -= gm.n[d]; ghost = true; }
        }
        src += (long)s * gm.st[d];
    }
    return src;
}
__device__ __forceinline__ void ghost_body(const Fields10 &f, const int nf, const Geom &gm, const long t)
{
    if (t >= gm.ntot) return;
    int idx[3];
    const long n = padded_node(gm, t, idx);
    bool ghost;
    const long src = periodic_image(gm, idx, ghost);
    if (!ghost) return;
#pragma unroll
    for (int m = 0; m < 10; m++)
        if (m < nf) f.f[m][n] = f.f[m][src];
}
__global__ void k_ghost_periodic(Fields10 f, int nf, Geom gm)
{
    ghost_body(f, nf, gm, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

// Sutherland viscosity at temperature ratio x.  x^1.5 as x sqrt(x): two roundings, like pow's result,
// at a tenth of its instructions (pow took 250 of the 390 k_ghost_values issues per node).
__device__ __forceinline__ double sutherland(const Consts &k, const double x)
{
    return (1.0 + k.suth) * (x * sqrt(x)) / (x + k.suth);
}

// ---- face boundary writers ---------------------------------------------------------------
// One launch per non-periodic face, in the reference's face order, after CalcValues.  A thread
// owns one ghost node of the face slab: layer l outside the face, tangential indices (i1, i2).
// Its mirror node is layer l inside the face (StartReal + l, EndReal - l).
// Cases with a subsonic outflow face keep the stored p and c of every node (P, C): CalcValues
// values, overwritten by every face writer on its ghosts.  Those writers store p and c that the
// equation of state does not give from rho,u,v,w,e, and the flux kernels read them there.
struct BcArgs {
    Fields5 pr;              // stage input state; ghost rho,u,v,w,e are written
    gdp T, mu;               // derived T and mu (viscous runs; null when inviscid)
    gcdp bs[6];              // exact rho,u,v,w,e,p for manufactured faces
    gcdp met[9];             // metric rows (subsonic outflow writers)
    gdp P, C;                // stored p and c (null unless a face is a subsonic outflow)
    gdp PL, RL, UL;          // Rudy: step-start ghost p, rho, u (written by face_save_body)
    gcdp C0;                 // Rudy: sound speed of the uploaded state
    int kind, dir, upper, g;
    int t1, t2;              // tangential axes
    int lo1, n1, lo2, n2;    // tangential index ranges
    int first, last;         // first / last interior index along dir
    long st[3];
    double rho_in, u_in, v_in, w_in, p_in, cinf, mach;
    double T_wall;           // isothermal walls
    double p_out, alpha_tau; // subsonic outflow: p_out and AlphaNonRef * tau
    Consts k;
};

// ghost node n and mirror node s of work item t of a face launch; false past the slab
__device__ __forceinline__ bool face_node(const BcArgs &a, const long t, long &n, long &s)
{
    const long per_layer = (long)a.n1 * a.n2;
    if (t >= per_layer * a.g) return false;
    const int l = (int)(t / per_layer);
    const long r = t - (long)l * per_layer;
    const int i1 = a.lo1 + (int)(r / a.n2), i2 = a.lo2 + (int)(r % a.n2);
    const int gi = a.upper ? a.last + 1 + l : a.first - 1 - l;
    const int si = a.upper ? a.last - l : a.first + l;
    const long base = (long)i1 * a.st[a.t1] + (long)i2 * a.st[a.t2];
    n = base + (long)gi * a.st[a.dir];
    s = base + (long)si * a.st[a.dir];
    return true;
}

// Rudy faces at the start of a step: U_lastStep's ghost p, rho and u, which the writers of every
// stage read (the first stage's writers overwrite the state buffer's ghosts)
__device__ __forceinline__ void face_save_body(const BcArgs &a, const long t)
{
    long n, s;
    if (!face_node(a, t, n, s)) return;
    a.PL[n] = a.P[n];
    a.RL[n] = a.pr.f[0][n];
    a.UL[n] = a.pr.f[1][n];
}

// contravariant velocities of the mirror node s (its CalcValues theta), the one along `flip`
// reversed (flip < 0: none), then the Cartesian velocity that has them under the metric rows of
// ghost node n: Cramer's rule, terms in the reference's order (src/BC.c:2556-2558, 2697-2699)
__device__ __forceinline__ void ghost_velocity(const BcArgs &a, const long n, const long s, const int flip,
                                               double &u, double &v, double &w)
{
    const double us = a.pr.f[1][s], vs = a.pr.f[2][s], ws = a.pr.f[3][s];
    double t0 = us * a.met[0][s] + vs * a.met[1][s] + ws * a.met[2][s];
    double t1 = us * a.met[3][s] + vs * a.met[4][s] + ws * a.met[5][s];
    double t2 = us * a.met[6][s] + vs * a.met[7][s] + ws * a.met[8][s];
    if (flip == 0) t0 = -t0;
    if (flip == 1) t1 = -t1;
    if (flip == 2) t2 = -t2;
    const double xx = a.met[0][n], xy = a.met[1][n], xz = a.met[2][n], ex = a.met[3][n], ey = a.met[4][n],
                 ez = a.met[5][n], zx = a.met[6][n], zy = a.met[7][n], zz = a.met[8][n];
    const double den = -xx * ey * zz + xx * ez * zy + xy * ex * zz - xy * ez * zx - xz * ex * zy + xz * ey * zx;
    u = -(t0 * ey * zz - t0 * ez * zy - t1 * xy * zz + t1 * xz * zy + t2 * xy * ez - t2 * xz * ey) / den;
    v = -(-t0 * ex * zz + t0 * ez * zx + t1 * xx * zz - t1 * xz * zx - t2 * xx * ez + t2 * xz * ex) / den;
    w = -(-t0 * ex * zy + t0 * ey * zx + t1 * xx * zy - t1 * xy * zx - t2 * xx * ey + t2 * xy * ex) / -den;
}

__device__ __forceinline__ void face_body(const BcArgs &a, const long t)
{
    long n, s;
    if (!face_node(a, t, n, s)) return;
    const Consts &k = a.k;
    if (a.kind == SHX_BC_WALL_SLIP || a.kind == SHX_BC_WALL_NOSLIP || a.kind == SHX_BC_WALL_ISOTHERMAL) {
        // WriteWallSlipBoundary (src/BC.c:2688-2719): the mirror's contravariant velocity along
        // the face's direction reversed; WriteWallNoSlipBoundary (src/BC.c:2657-2686): all
        // velocities reversed.  rho, e, p, c, T and mu from the mirror node.  The corrector these
        // writers store is applied by the WENO sweeps on the ghost nodes of wall faces.
        double u, v, w;
        if (a.kind == SHX_BC_WALL_SLIP) {
            ghost_velocity(a, n, s, a.dir, u, v, w);
        } else {
            u = -a.pr.f[1][s]; v = -a.pr.f[2][s]; w = -a.pr.f[3][s];
        }
        a.pr.f[0][n] = a.pr.f[0][s]; a.pr.f[1][n] = u; a.pr.f[2][n] = v; a.pr.f[3][n] = w;
        a.pr.f[4][n] = a.pr.f[4][s];
        if (a.P) { a.P[n] = a.P[s]; a.C[n] = a.C[s]; }
        // WriteWallNoSlipIsothermalBoundary (src/BC.c:2943-2978): T = T_wall on the ghost
        if (a.T) { a.T[n] = (a.kind == SHX_BC_WALL_ISOTHERMAL) ? a.T_wall : a.T[s]; a.mu[n] = a.mu[s]; }
        return;
    }
    if (a.kind == SHX_BC_OUTFLOW_NORMAL || a.kind == SHX_BC_OUTFLOW_RUDY) {
        double u, v, w;
        ghost_velocity(a, n, s, -1, u, v, w);
        double p, rho;
        if (a.kind == SHX_BC_OUTFLOW_RUDY) {
            p = (a.PL[n] + a.alpha_tau * a.p_out + a.RL[n] * a.C0[s] * (u - a.UL[n]) / k.upsilon) / (1.0 + a.alpha_tau);
            rho = p / a.P[s] * a.pr.f[0][s];
        } else {
            p = a.p_out;
            rho = a.pr.f[0][s];
        }
        a.pr.f[0][n] = rho; a.pr.f[1][n] = u; a.pr.f[2][n] = v; a.pr.f[3][n] = w;
        a.pr.f[4][n] = a.pr.f[4][s];
        a.P[n] = p;
        a.C[n] = a.C[s];
        if (a.T) { a.T[n] = a.T[s]; a.mu[n] = a.mu[s]; }
        return;
    }
    if (a.kind == SHX_BC_FARFIELD) {
        // WriteFarfieldBoundary (src/BC.c:2817-2852): the mirror node's values
#pragma unroll
        for (int m = 0; m < 5; m++) a.pr.f[m][n] = a.pr.f[m][s];
        if (a.P) { a.P[n] = a.P[s]; a.C[n] = a.C[s]; }
        if (a.T) { a.T[n] = a.T[s]; a.mu[n] = a.mu[s]; }
        return;
    }
    if (a.kind == SHX_BC_INFLOW_SUB_NORMAL || a.kind == SHX_BC_INFLOW_SUB_RIEMANN ||
        a.kind == SHX_BC_INFLOW_SUB_ISENTROPIC) {
        // subsonic inflow (src/BC.c:2363-2503): velocity, rho and p by the writer's rule, e and c
        // from them, T and mu from the mirror node
        const double gm = k.gamma;
        double u, v, w, rho, p;
        if (a.kind == SHX_BC_INFLOW_SUB_NORMAL) {
            u = a.u_in; v = a.v_in; w = a.w_in;
            p = a.p_in; rho = a.rho_in;
        } else if (a.kind == SHX_BC_INFLOW_SUB_RIEMANN) {
            // incoming invariant and entropy of the far field, outgoing invariant of the mirror
            const double rs = a.pr.f[0][s], us = a.pr.f[1][s];
            const double cii = a.P ? a.C[s]
                                   : sqrt(k.upsilon * gm * pressure(k, rs, us, a.pr.f[2][s], a.pr.f[3][s], a.pr.f[4][s]) / rs);
            u = 0.5 * (us + a.u_in) + (a.cinf - cii) / (gm - 1.);
            v = a.v_in; w = a.w_in;
            const double d1 = (0.5 * (cii + a.cinf) + 0.25 * (gm - 1.) * (a.u_in - us)) / a.cinf;
            rho = a.rho_in * pow(d1, 2. / (gm - 1.));
            p = a.p_in * pow(d1, 2. * gm / (gm - 1.));
        } else {
            // the mirror's contravariant velocities, rho from Bernoulli along the far field's isentrope
            ghost_velocity(a, n, s, -1, u, v, w);
            rho = pow(pow(a.rho_in, (gm - 1.0)) - pow(a.rho_in, gm) / a.p_in * (gm - 1.0) / gm * gm * a.mach * a.mach
                      * (u * u / 2.0), 1.0 / (gm - 1.0));
            p = a.p_in * pow(rho / a.rho_in, gm);
        }
        a.pr.f[0][n] = rho; a.pr.f[1][n] = u; a.pr.f[2][n] = v; a.pr.f[3][n] = w;
        a.pr.f[4][n] = (0.5 * ((u * u) + (v * v) + (w * w)) + p / rho / (gm - 1.0) * k.upsilon);
        if (a.T) { a.T[n] = a.T[s]; a.mu[n] = a.mu[s]; }
        if (a.P) { a.P[n] = p; a.C[n] = sqrt(k.upsilon * gm * p / rho); }
        return;
    }
    if (a.kind == SHX_BC_MANUFACTURED) {
        // WriteManufacturedSolution: exact state, T = |p/rho|, mu = 1 (c, p and theta are
        // recomputed from rho,u,v,w,e where the flux kernels need them)
        const double rho = a.bs[0][n];
        for (int m = 0; m < 5; m++) a.pr.f[m][n] = a.bs[m][n];
        if (a.T) { a.T[n] = fabs(a.bs[5][n] / rho); a.mu[n] = 1.0; }
        if (a.P) { a.P[n] = a.bs[5][n]; a.C[n] = sqrt(k.upsilon * k.gamma * a.bs[5][n] / rho); }
    } else if (a.kind == SHX_BC_INFLOW_SUPERSONIC) {
        const double rho = a.rho_in, u = a.u_in, v = a.v_in, w = a.w_in, p = a.p_in;
        a.pr.f[0][n] = rho; a.pr.f[1][n] = u; a.pr.f[2][n] = v; a.pr.f[3][n] = w;
        a.pr.f[4][n] = (0.5 * ((u * u) + (v * v) + (w * w)) + p / rho / (k.gamma - 1.0) * k.upsilon);
        if (a.T) {
            a.T[n] = a.p_in / a.rho_in;
            a.mu[n] = sutherland(k, p / rho);
        }
        if (a.P) { a.P[n] = p; a.C[n] = sqrt(k.upsilon * k.gamma * p / rho); }
    } else {
        // Riemann invariants: outgoing from the mirror node, incoming from the inflow state
        const double rs = a.pr.f[0][s], us = a.pr.f[1][s], vs = a.pr.f[2][s], ws = a.pr.f[3][s];
        const double ps = a.P ? a.P[s] : pressure(k, rs, us, vs, ws, a.pr.f[4][s]);
        const double cii = a.P ? a.C[s] : sqrt(k.upsilon * k.gamma * ps / rs);
        const double u = 0.5 * (us + a.u_in) - (a.cinf - cii) / (k.gamma - 1.);
        const double d1 = (0.5 * (cii + a.cinf) - 0.25 * (k.gamma - 1.) * (a.u_in - us)) / cii;
        const double rho = rs * pow(d1, 2. / (k.gamma - 1.));
        const double p = ps * pow(d1, 2. * k.gamma / (k.gamma - 1.));
        a.pr.f[0][n] = rho; a.pr.f[1][n] = u; a.pr.f[2][n] = vs; a.pr.f[3][n] = ws;
        a.pr.f[4][n] = (0.5 * ((u * u) + (vs * vs) + (ws * ws)) + p / rho / (k.gamma - 1.0) * k.upsilon);
        if (a.T) { a.T[n] = a.T[s]; a.mu[n] = a.mu[s]; }
        if (a.P) { a.P[n] = p; a.C[n] = sqrt(k.upsilon * k.gamma * p / rho); }
    }
}
// mirrorGhostCellsMetric (src/Functions.c:6849-7014): every ghost node of a wall or farfield face's
// slab (the whole tangential range) takes the metric of its mirror node
__global__ void k_mirror_metric(BcArgs a, Fields10 met)
{
    long n, s;
    if (!face_node(a, (long)blockIdx.x * blockDim.x + threadIdx.x, n, s)) return;
#pragma unroll
    for (int m = 0; m < 10; m++) met.f[m][n] = met.f[m][s];
}
__global__ void k_face_save(BcArgs a)
{
    face_save_body(a, (long)blockIdx.x * blockDim.x + threadIdx.x);
}
__global__ void k_face_bc(BcArgs a)
{
    face_body(a, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

// Ghost nodes of non-periodic directions carried from one stage buffer to the next: the
// reference keeps one U_RK array whose ghost layers persist between stages, which matters where
// a writer reads a ghost another face wrote in the previous stage.
__device__ __forceinline__ void carry_body(const CFields5 &from, const Fields5 &to, const Geom &gm, const long t)
{
    if (t >= gm.ntot) return;
    int idx[3];
    const long n = padded_node(gm, t, idx);
    bool ghost = false;
#pragma unroll
    for (int d = 0; d < 3; d++)
        if (gm.ng[d] > 1 && !gm.per[d] && (idx[d] < gm.lo[d] || idx[d] >= gm.lo[d] + gm.n[d])) ghost = true;
    if (!ghost) return;
#pragma unroll
    for (int m = 0; m < 5; m++) to.f[m][n] = from.f[m][n];
}
__global__ void k_carry_ghosts(CFields5 from, Fields5 to, Geom gm)
{
    carry_body(from, to, gm, (long)blockIdx.x * blockDim.x + threadIdx.x);
}
// every ghost node (periodic directions included) copied from one buffer to another; image: from its
// periodic image there (all directions periodic: what a ghost fill of that buffer holds)
__global__ void k_copy_ghosts(CFields5 from, Fields5 to, Geom gm, int image)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= gm.ntot) return;
    int idx[3];
    const long n = padded_node(gm, t, idx);
    bool ghost = false;
#pragma unroll
    for (int d = 0; d < 3; d++)
        if (gm.ng[d] > 1 && (idx[d] < gm.lo[d] || idx[d] >= gm.lo[d] + gm.n[d])) ghost = true;
    if (!ghost) return;
    long src = n;
    if (image) src = periodic_image(gm, idx, ghost);
#pragma unroll
    for (int m = 0; m < 5; m++) to.f[m][n] = from.f[m][src];
}

// T = |p/rho| and mu (Sutherland, or 1 under the manufactured solution) of one node, CalcValues
// (src/Functions.c:2462-2476)
__device__ __forceinline__ void node_tmu(const Consts &k, const double p, const double rho, double &T, double &mu)
{
    T = fabs(p / rho);
    mu = k.mms ? 1.0 : sutherland(k, p / rho);
}

// T and mu of node n (viscous runs), and its stored p and c (cases with a subsonic outflow face)
__device__ __forceinline__ void node_values(const double rho, const double u, const double v, const double w,
                                            const double e, const gdp T, const gdp mu, const gdp P, const gdp C,
                                            const Consts &k, const long n)
{
    const double p = pressure(k, rho, u, v, w, e);
    if (T) {
        double t, m;
        node_tmu(k, p, rho, t, m);
        T[n] = t;
        mu[n] = m;
    }
    if (P) { P[n] = p; C[n] = sqrt(k.upsilon * k.gamma * p / rho); }
}
// CalcValues on all padded nodes
__device__ __forceinline__ void values_body(const CFields5 &pr, const gdp T, const gdp mu, const gdp P,
                                            const gdp C, const Geom &gm, const Consts &k, const long t)
{
    if (t >= gm.ntot) return;
    int idx[3];
    const long n = padded_node(gm, t, idx);
    node_values(pr.f[0][n], pr.f[1][n], pr.f[2][n], pr.f[3][n], pr.f[4][n], T, mu, P, C, k, n);
}
// Periodic ghost fill of the primitives and CalcValues in one pass: a ghost node copies its
// periodic image and evaluates the values from the copied primitives, which gives the bits of the
// fill followed by CalcValues.  Only ghost nodes are written to pr, and they are never an image,
// so no thread reads a node another thread writes.
__device__ __forceinline__ void ghost_values_body(const Fields5 &pr, const gdp T, const gdp mu, const gdp P,
                                                  const gdp C, const Geom &gm, const Consts &k, const long t)
{
    if (t >= gm.ntot) return;
    int idx[3];
    const long n = padded_node(gm, t, idx);
    bool ghost;
    const long src = periodic_image(gm, idx, ghost);
    double q[5];
#pragma unroll
    for (int m = 0; m < 5; m++) q[m] = pr.f[m][src];
    if (ghost) {
#pragma unroll
        for (int m = 0; m < 5; m++) pr.f[m][n] = q[m];
    }
    node_values(q[0], q[1], q[2], q[3], q[4], T, mu, P, C, k, n);
}
__global__ void k_calc_values(CFields5 pr, gdp T, gdp mu, gdp P, gdp C, Geom gm, Consts k)
{
    values_body(pr, T, mu, P, C, gm, k, (long)blockIdx.x * blockDim.x + threadIdx.x);
}
__global__ void k_ghost_values(Fields5 pr, gdp T, gdp mu, gdp P, gdp C, Geom gm, Consts k)
{
    ghost_values_body(pr, T, mu, P, C, gm, k, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

// ---- block placement ------------------------------------------------------------------------
// Blocks are dispatched round-robin over the eight XCDs (block p on XCD p % 8), each with its own
// L2.  xcd_order hands XCD x a contiguous range of tiles in dispatch order, so tiles next to each
// other in the tile order (which share halo nodes) run on one L2 at about the same time.
__device__ __forceinline__ int xcd_order(const int p, const int total)
{
    const int per = total >> 3, rem = total & 7, x = p & 7, s = p >> 3;
    return x * per + min(x, rem) + s;
}
// Tile of block p; tg = (A tiles, B tiles, sweep tiles, order).  order 1: sweep tiles fastest,
// then A, then B, placed by xcd_order (neighbours along the sweep share halo nodes in one L2);
// order 0: A fastest in launch order, which keeps the row segments that consecutive blocks read
// adjacent in memory (measured faster where the sweep axis is the slowest one in memory).
__device__ __forceinline__ void sweep_tile(const int p, const int tg[4], int &bx, int &by, int &bz)
{
    if (tg[3] == 0) {
        bx = p % tg[0];
        by = (p / tg[0]) % tg[1];
        bz = p / (tg[0] * tg[1]);
        return;
    }
    const int q = xcd_order(p, tg[0] * tg[1] * tg[2]);
    bz = q % tg[2];
    const int r = q / tg[2];
    bx = r % tg[0];
    by = r / tg[0];
}

// ---- WENO sweep ---------------------------------------------------------------------------
struct WenoArgs {
    CFields5 pr;          // rho, u, v, w, e of the stage input (ghosts filled unless wrap)
    gcdp m0, m1, m2, J;               // metric row of the sweep direction and the Jacobian
                                      // (diagonal metrics: m0 is the row's diagonal entry)
    Fields5 q;            // stage residual, interior nodes
    gcdp P, C;            // stored p and c, read on the ghost nodes of subsonic outflow faces
    int pc_lo, pc_hi;     // the lower / upper face of the sweep direction stores p and c on its ghosts
    int w_lo, w_hi;       // the lower / upper face of the sweep direction is a wall
    double c_lo[3], c_hi[3];  // its corrector of the convective momentum terms (src/WENO.c:265-277)
    int tg[4];            // tile grid (A tiles, B tiles, sweep tiles) and order of a single-case launch
    long sD, sA, sB;      // strides: sweep, fast transverse, slow transverse
    int nD, nA, nB;       // interior counts
    int oD, oA, oB;       // padded index of the first interior node per axis
    int ngD;              // padded extent along the sweep
    int first;            // 1: Q = -div (first direction of the stage), 0: Q -= div
    int coalesce_d;       // load mapping: 1 when the sweep axis is contiguous in memory
    int alignA;           // tiles start at padded A index 0 (A axis contiguous, pitch padded)
    int wrap;             // the stage input's ghosts are read at their periodic image (state_wraps)
    Consts k;
};

// per-node values staged in LDS
enum { V_F0, V_F1, V_F2, V_F3, V_F4, V_U0, V_U1, V_U2, V_U3, V_U4, V_LAM, V_U, V_V, V_W, V_C,
       V_NX, V_NY, V_NZ, V_J, NV };

// AX = -1: general metric rows; AX = 0, 1, 2: diagonal metric, the sweep's normal is the axis AX
// (the reference's 3D metric, src/Functions.c:6479-6484), which drops two metric loads, two LDS
// fields and the zero entries of the eigenvector rows.
// MIX: mixed-precision form.  Node fluxes, the central part Theta, the eigen-system and the
// divergence stay FP64; the characteristic projection (of node-to-node differences of F and U,
// formed in FP64 and rounded once), the smoothness indicators, weights and the deviation Phi, and
// R . Phi are FP32.  Phi is a correction on top of Theta, so its rounding enters at the size of
// the correction rather than of the flux.
// LDS of one WENO sweep block, in doubles: the node window (NVK fields) and, in the mixed form,
// room for two of the ten FP32 difference arrays (the other eight reuse four conserved-variable
// fields of the window).  Diagonal metric: no normal components; the sign of the
// metric entry rides on V_LAM (the spectral radius is positive) and J moves to V_NX, which keeps
// the 8 x 32 tile's window under 40 KB (four blocks per CU).
template <int S, int TA, int TDI, int AX, bool MIX>
constexpr int weno_lds()
{
    constexpr int NW = (TDI - 1 + (S + 1)) * TA;
    constexpr int NVK = (AX < 0) ? NV : NV - 3;
    return NVK * NW + (MIX ? NW : 0);
}

// Value of the next lane (lane 63: its own).  All 64 lanes must be active.
__device__ __forceinline__ double next_lane(const double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = (int)b, hi = (int)(b >> 32);
    const int nlo = __builtin_amdgcn_update_dpp(lo, lo, 0x130, 0xf, 0xf, false);   // wave_shl:1
    const int nhi = __builtin_amdgcn_update_dpp(hi, hi, 0x130, 0xf, 0xf, false);
    return __longlong_as_double(((long long)nhi << 32) | (unsigned)nlo);
}

// FP64 WENO flux of the interface between nodes ob+R and ob+R+1 of a window row (R = G-1), less
// F[ob+R]: the central part in differences D[j] = F[ob+R+j+1] - F[ob+R+j],
//   Theta - F = (D[-1] + 6 D[0] - D[1]) / 12                                              (WENO5)
//             = (420 D[0] + 113 (D[-1]-D[1]) - 26 (D[-2]-D[2]) + 3 (D[-3]-D[3])) / 840     (WENO9),
// whose F terms telescope in the divergence (the upper node's divergence = D[0], returned in dcur,
// plus the difference of the two interface values), and R Phi.
// The nodes pass through registers once: a pair of neighbours gives its differences of F and U, the
// split differences dF +- lam J dU, and their five characteristic projections (char_project), so the
// window is read 80 to 120 times per WENO5 interface instead of 190 (once per non-zero entry of the
// left eigenvectors), which had the LDS as busy as the FP64 pipe, and FP64 instructions fall from 926
// to about 750 (256^3, diagonal metric: xi sweep 1.04 -> 0.82 ms, k_eta 1.42 -> 1.26, k_zeta 1.70 -> 1.57).
// WENO9, 176 x 128 x 136: xi and eta sweeps 425 and 457 -> 309 and 327 us, k_zeta 684 -> 523 (447 on its 8 x 32
// tile; indicators as sums of squares of the differences, w9_is, and three waves per SIMD instead of two).
// Bound by the FP64 pipe and its latency, so registers decide: the projections are pinned pair by pair
// (else the compiler keeps several pairs in flight, 148-166 VGPRs for WENO5), which leaves WENO5 along
// zeta 128 VGPRs, four waves per SIMD.  Along xi and eta one pass over all fields still spilled two
// registers (k_eta 1.31 ms), so they take the shear fields, which need three of the five components,
// in a second pass over the row; so does WENO9 everywhere, for three waves.
template <int S, int AX, int NW, int VJ>
__device__ __forceinline__ void weno_flux(const double *sm, const int ob, const Consts &k, double out[5], double dcur[5])
{
    constexpr int R = (S - 1) / 2;
    const int oc = ob + R;
    auto mean = [&](const int v) { return 0.5 * (sm[v * NW + oc] + sm[v * NW + oc + 1]); };
    const double cs = mean(V_C);
    const double rho = mean(V_U0);
    CharBasis c;
    c.u[0] = mean(V_U); c.u[1] = mean(V_V); c.u[2] = mean(V_W);
    if constexpr (AX < 0) {
        c.n[0] = mean(V_NX); c.n[1] = mean(V_NY); c.n[2] = mean(V_NZ);
    } else {
        c.s = 0.5 * (copysign(1.0, sm[V_LAM * NW + oc]) + copysign(1.0, sm[V_LAM * NW + oc + 1]));
    }
    char_basis<AX>(c, rho, cs, k.gamma);
    double lam = 0.0;
#pragma unroll
    for (int s = 0; s < S + 1; s++) lam = fmax(lam, fabs(sm[V_LAM * NW + ob + s]));
    const double lj = lam * mean(VJ);

    // epsilon of the indicators as w5_pair and w9_pair form them, scaled with the square of what the
    // projections leave out (char_project)
    const double e0 = (S == 5) ? k.eps * (1. / 3.) : k.eps;
    const double es = (AX < 0) ? e0 : e0 * (rho * rho), ea = 2.0 * e0;
    double psi[5];
    // one pass over the row's pairs for the fields of MASK (bit f: field f)
    auto pass = [&](auto mask_c) {
        constexpr int MASK = decltype(mask_c)::value;
        double fp[5][S - 1], fm[5][S - 1];       // split characteristic differences: f+ of pairs 0..S-2, f- of S-1..1
        double pf[5], pu[5];
        // components the fields need: all, or mass and the transverse momenta for the shear fields
        auto need = [](const int q) { return AX < 0 || (MASK & 25) || (q != 1 + AX && q != 4); };
#pragma unroll
        for (int q = 0; q < 5; q++)
            if (need(q)) { pf[q] = sm[(V_F0 + q) * NW + ob]; pu[q] = sm[(V_U0 + q) * NW + ob]; }
#pragma unroll
        for (int s = 0; s < S; s++) {
            double dF[5] = {}, dU[5] = {};
#pragma unroll
            for (int q = 0; q < 5; q++) {
                if (!need(q)) continue;
                const double f = sm[(V_F0 + q) * NW + ob + s + 1], u = sm[(V_U0 + q) * NW + ob + s + 1];
                dF[q] = f - pf[q]; dU[q] = u - pu[q];
                pf[q] = f; pu[q] = u;
            }
            double g[5], o[5];
            if (s < S - 1) {
#pragma unroll
                for (int q = 0; q < 5; q++) g[q] = fma(lj, dU[q], dF[q]);
                char_project<AX>(c, g, o);
#pragma unroll
                for (int f = 0; f < 5; f++) if (MASK >> f & 1) fp[f][s] = o[f];
            }
            if (s > 0) {
#pragma unroll
                for (int q = 0; q < 5; q++) g[q] = fma(-lj, dU[q], dF[q]);
                char_project<AX>(c, g, o);
#pragma unroll
                for (int f = 0; f < 5; f++) if (MASK >> f & 1) fm[f][S - 1 - s] = o[f];
            }
            // one pair's loads and projections at a time (registers)
#pragma unroll
            for (int f = 0; f < 5; f++) {
                if (!(MASK >> f & 1)) continue;
                if (s < S - 1) asm volatile("" : "+v"(fp[f][s]));
                if (s > 0) asm volatile("" : "+v"(fm[f][S - 1 - s]));
            }
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int f = 0; f < 5; f++) {
            if (!(MASK >> f & 1)) continue;
            const double e = (f >= 3) ? ea : (f ? es : e0);
            if constexpr (S == 5) psi[f] = w5_pair(e, fp[f], fm[f]);
            else psi[f] = w9_pair(e, fp[f], fm[f]);
        }
    };
    if constexpr (S == 9 && AX < 0) {
        pass(std::integral_constant<int, 24>{});
        asm volatile("" : "+v"(psi[3]), "+v"(psi[4]) : : "memory");
        pass(std::integral_constant<int, 7>{});
    } else if constexpr (S == 9 || AX == 0 || AX == 1) {
        pass(std::integral_constant<int, 25>{});
        asm volatile("" : "+v"(psi[0]), "+v"(psi[3]), "+v"(psi[4]) : : "memory");
        pass(std::integral_constant<int, 6>{});
    } else {
        pass(std::integral_constant<int, 31>{});
    }
    char_assemble<AX>(c, rho, cs * cs * k.igm1, psi, out);
#pragma unroll
    for (int m = 0; m < 5; m++) {
        const double *F = &sm[(V_F0 + m) * NW + oc];
        const double d0 = F[1] - F[0];
        const double a1 = (F[0] - F[-1]) - (F[2] - F[1]);
        if constexpr (S == 5) {
            out[m] += 1. / 12. * (a1 + 6. * d0);
        } else {
            const double a2 = (F[-1] - F[-2]) - (F[3] - F[2]), a3 = (F[-2] - F[-3]) - (F[4] - F[3]);
            out[m] += 1. / 840. * (420. * d0 + 113. * a1 - 26. * a2 + 3. * a3);
        }
        dcur[m] = d0;
    }
}

// KEEP: leave Q alone and return this sweep's contribution of the thread's node in keep[5] (a
// fused kernel adds it later); otherwise Q = -div (first sweep of the stage) or Q -= div.
// NT: threads that sweep the tile together, a multiple of the wavefront not below TA * TDI (those past it
// repeat the last row); a group of NT threads within a larger block.
template <int S, int TA, int TDI, int AX, bool MIX, bool KEEP = false, int NT = TA * TDI>
__device__ __forceinline__ void weno_body(const WenoArgs &a, const int bx, const int by, const int bz,
                                          double *lds, double *keep = nullptr)
{
    constexpr int G = (S + 1) / 2;
    constexpr int R = G - 1;
    constexpr int WD = TDI - 1 + 2 * G;   // window nodes along the sweep
    constexpr int NW = WD * TA;
    constexpr int NVK = (AX < 0) ? NV : NV - 3;
    constexpr int VJ = (AX < 0) ? V_J : V_NX;
    constexpr int NMET = (AX < 0) ? 3 : 1;
    // the FP64 form streams the stencil through registers pair by pair (weno_flux); the mixed form
    // projects one characteristic field at a time
    constexpr bool PAIRS = !MIX;
    // the plus-side interface value of a node's divergence comes from the next lane where a tile row
    // never straddles two wavefronts
    constexpr bool SHFL = (64 % TDI == 0);
    double *const sm = lds;                       // NVK * NW (+ NW)
    // mixed form: the FP32 differences of F (arrays 0..4) and U (5..9).  Once formed, the node
    // values of rho u, rho v, rho w and rho e are not read again, so arrays 0..7 take their place
    // (V_U1..V_U4) and only arrays 8 and 9 extend the window: the 8 x 32 tile keeps four blocks
    // per CU.
    auto dfa = [&](const int j) -> float * {
        return (j < 8) ? (float *)(lds + V_U1 * NW) + j * NW : (float *)(lds + NVK * NW) + (j - 8) * NW;
    };

    const int t = (NT == TA * TDI) ? threadIdx.x : threadIdx.x % NT;
    // first padded A index of the tile (aligned to TA when the A axis is contiguous in memory)
    const int pa0 = a.alignA ? bx * TA : bx * TA + a.oA;
    const int b = by;
    const int d0 = bz * (TDI - 1);               // first node of this tile (interior-relative)
    const long bbase = (long)(b + a.oB) * a.sB;
    const Consts &k = a.k;

    // phase 1: per-node flux, conserved vector, spectral radius and eigenvector inputs.  Sweeps
    // of a direction with a wall face take a second copy of the loop (WALL), so the others keep
    // the plain node flux.
    auto node_pass = [&](auto wall_c) {
    constexpr bool WALL = decltype(wall_c)::value;
    constexpr int PER = (NW + NT - 1) / NT;
    // the loads of all rounds first: the last round is one wavefront's, and the others wait for it at the
    // barrier (256^3, k_zeta 1.57 -> 1.50 ms FP64, 1.64 -> 1.53 mixed)
    double in[PER][6 + NMET];
    long nn[PER];
    int dpr[PER], op[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int idx = t + r * NT;
        if (idx >= NW) continue;
        int aa, dd;
        if (a.coalesce_d) { aa = idx / WD; dd = idx - aa * WD; }
        else { dd = idx / TA; aa = idx - dd * TA; }
        const int pa = max(a.oA, min(pa0 + aa, a.oA + a.nA - 1));
        int dp = d0 - G + dd + a.oD;
        dp = max(0, min(dp, a.ngD - 1));
        const long n = bbase + (long)pa * a.sA + (long)dp * a.sD;
        // wrap: a ghost node of the stage input is read at its periodic image
        long ns = n;
        if (a.wrap) ns += (long)(dp < a.oD ? a.nD : (dp >= a.oD + a.nD ? -a.nD : 0)) * a.sD;
#pragma unroll
        for (int m = 0; m < 5; m++) in[r][m] = a.pr.f[m][ns];
        in[r][5] = a.J[n];
        in[r][6] = a.m0[n];
        if constexpr (AX < 0) { in[r][7] = a.m1[n]; in[r][8] = a.m2[n]; }
        nn[r] = n; dpr[r] = dp; op[r] = aa * WD + dd;
    }
#pragma unroll
    for (int r = 0; r < PER; r++) {
        if (t + r * NT >= NW) continue;
        const long n = nn[r];
        const int dp = dpr[r], o = op[r];
        const double rho = in[r][0], u = in[r][1], v = in[r][2], w = in[r][3], e = in[r][4], J = in[r][5];
        double p = pressure_fast(k, rho, u, v, w, e);
        const double ir = frcp(rho);
        double cs = sqrt(k.upsilon * k.gamma * p * ir);
        if ((a.pc_lo && dp < a.oD) || (a.pc_hi && dp >= a.oD + a.nD)) { p = a.P[n]; cs = a.C[n]; }
        const double pu = p * k.upsilon;
        // velocities of the convective momentum terms: times the wall corrector (+-1, exact) on
        // the ghost nodes of a wall face of this direction, the velocities themselves elsewhere
        double uc[3] = {u, v, w};
        if constexpr (WALL) {
            if ((a.w_lo && dp < a.oD) || (a.w_hi && dp >= a.oD + a.nD)) {
                const bool lo = dp < a.oD;
#pragma unroll
                for (int q = 0; q < 3; q++) uc[q] *= lo ? a.c_lo[q] : a.c_hi[q];
            }
        }
        if constexpr (AX < 0) {
            const double mx = in[r][6], my = in[r][7], mz = in[r][8];
            const double th = u * mx + v * my + w * mz;
            const double rt = rho * th;
            sm[V_F0 * NW + o] = J * rt;
            sm[V_F1 * NW + o] = J * (rt * uc[0] + mx * pu);
            sm[V_F2 * NW + o] = J * (rt * uc[1] + my * pu);
            sm[V_F3 * NW + o] = J * (rt * uc[2] + mz * pu);
            sm[V_F4 * NW + o] = J * (rt * (e + pu * ir));
            const double mn = sqrt(mx * mx + my * my + mz * mz);
            const double imn = frcp(mn);
            sm[V_LAM * NW + o] = fabs(th) + cs * mn;
            sm[V_NX * NW + o] = mx * imn;
            sm[V_NY * NW + o] = my * imn;
            sm[V_NZ * NW + o] = mz * imn;
        } else {
            const double md = in[r][6];
            const double uu[3] = {u, v, w};
            const double th = uu[AX] * md;
            const double rt = rho * th;
            sm[V_F0 * NW + o] = J * rt;
#pragma unroll
            for (int q = 0; q < 3; q++) sm[(V_F1 + q) * NW + o] = (q == AX) ? J * (rt * uc[q] + md * pu) : J * (rt * uc[q]);
            sm[V_F4 * NW + o] = J * (rt * (e + pu * ir));
            const double lam = fabs(th) + cs * fabs(md);
            sm[V_LAM * NW + o] = (md > 0.0) ? lam : -lam;
        }
        sm[V_U0 * NW + o] = rho;
        sm[V_U1 * NW + o] = rho * u;
        sm[V_U2 * NW + o] = rho * v;
        sm[V_U3 * NW + o] = rho * w;
        sm[V_U4 * NW + o] = rho * e;
        sm[V_U * NW + o] = u;
        sm[V_V * NW + o] = v;
        sm[V_W * NW + o] = w;
        sm[V_C * NW + o] = cs;
        sm[VJ * NW + o] = J;
    }
    };
    if (a.w_lo || a.w_hi) node_pass(std::true_type{});
    else node_pass(std::false_type{});
    __syncthreads();
    if constexpr (MIX) {
        // node-to-node differences of F and U, rounded once to FP32 (position o: node o+1 - node o),
        // all read before any is written over the conserved values
        constexpr int PER = (NW + NT - 1) / NT;
        float dv[PER][10];
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int idx = t + r * NT;
            if (idx < NW && idx % WD != WD - 1) {
#pragma unroll
                for (int q = 0; q < 5; q++) {
                    dv[r][q] = (float)(sm[(V_F0 + q) * NW + idx + 1] - sm[(V_F0 + q) * NW + idx]);
                    dv[r][5 + q] = (float)(sm[(V_U0 + q) * NW + idx + 1] - sm[(V_U0 + q) * NW + idx]);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int idx = t + r * NT;
            if (idx < NW && idx % WD != WD - 1) {
#pragma unroll
                for (int j = 0; j < 10; j++) dfa(j)[idx] = dv[r][j];
            }
        }
        __syncthreads();
    }

    // phase 2: interface flux between nodes (d0-1+di) and (d0+di)
    const int ta = (NT == TA * TDI) ? t / TDI : min(t / TDI, TA - 1), di = t % TDI;
    const int ob = ta * WD + di;                 // window position of the stencil's first node
    const int oc = ob + R;                       // left node of the interface
    double out[5];
    double dcur[5];                              // PAIRS: F[oc+1] - F[oc], for the divergence
    if constexpr (PAIRS) {
        weno_flux<S, AX, NW, VJ>(sm, ob, k, out, dcur);
    } else {
        const double Jh = (sm[VJ * NW + oc] + sm[VJ * NW + oc + 1]) / 2.0;
        const double u = 0.5 * (sm[V_U * NW + oc] + sm[V_U * NW + oc + 1]);
        const double v = 0.5 * (sm[V_V * NW + oc] + sm[V_V * NW + oc + 1]);
        const double w = 0.5 * (sm[V_W * NW + oc] + sm[V_W * NW + oc + 1]);
        const double rho = 0.5 * (sm[V_U0 * NW + oc] + sm[V_U0 * NW + oc + 1]);
        const double cs = 0.5 * (sm[V_C * NW + oc] + sm[V_C * NW + oc + 1]);
        double nx, ny, nz;
        if constexpr (AX < 0) {
            nx = 0.5 * (sm[V_NX * NW + oc] + sm[V_NX * NW + oc + 1]);
            ny = 0.5 * (sm[V_NY * NW + oc] + sm[V_NY * NW + oc + 1]);
            nz = 0.5 * (sm[V_NZ * NW + oc] + sm[V_NZ * NW + oc + 1]);
        } else {
            const double ns = 0.5 * (copysign(1.0, sm[V_LAM * NW + oc]) + copysign(1.0, sm[V_LAM * NW + oc + 1]));
            nx = (AX == 0) ? ns : 0.0;
            ny = (AX == 1) ? ns : 0.0;
            nz = (AX == 2) ? ns : 0.0;
        }
        const double nsig = (AX == 0) ? nx : ((AX == 1) ? ny : nz);
        const Eig e = make_eig(nx, ny, nz, u, v, w, rho, cs, k.gamma);
        double lam = 0.0;
#pragma unroll
        for (int s = 0; s < 2 * G; s++) lam = fmax(lam, (AX < 0) ? sm[V_LAM * NW + ob + s] : fabs(sm[V_LAM * NW + ob + s]));
        const double lj = lam * Jh;

        // Characteristic projection per field c: a_s = L_c . F_s and b_s = L_c . U_s on the 2G
        // stencil nodes, f+_s = (a_s + lam J b_s)/2 on nodes m-r..m+r and f-_s = (a - lam J b)/2
        // on the mirrored nodes m+r+1..m-r+1 (src/WENO.c:334-385).
        float phif[5];
        auto project = [&](auto cc) {
            constexpr int c = decltype(cc)::value;
            double Ld[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            if constexpr (AX < 0) left_row<c>(e, Ld);
            else left_row_ax<c, (AX < 0 ? 0 : AX)>(e, nsig, Ld);
            float Lf[5];
#pragma unroll
            for (int q = 0; q < 5; q++) Lf[q] = (float)Ld[q];
            const float ljf = (float)lj;
            // projected differences da_s = L_c . (F_{s+1} - F_s), db_s likewise for U
            float dp[S - 1], dm[S - 1];
            float da[2 * G - 1], db[2 * G - 1];
#pragma unroll
            for (int s = 0; s < 2 * G - 1; s++) {
                float x = 0.f, y = 0.f;
#pragma unroll
                for (int q = 0; q < 5; q++) {
                    if (AX < 0 || lnz(c, AX, q)) {
                        x += Lf[q] * dfa(q)[ob + s];
                        y += Lf[q] * dfa(5 + q)[ob + s];
                    }
                }
                da[s] = x;
                db[s] = y;
            }
            // differences of the split fluxes (times 2, see below): f+ on nodes 0..S-1, f- mirrored
#pragma unroll
            for (int s = 0; s < S - 1; s++) {
                dp[s] = da[s] + ljf * db[s];
                dm[s] = da[S - 1 - s] - ljf * db[S - 1 - s];
            }
            if constexpr (S == 5) {
                phif[c] = 0.5f * (-phi_w5_f(dp[0], dp[1], dp[2], dp[3]) + phi_w5_f(dm[0], dm[1], dm[2], dm[3]));
            } else {
                phif[c] = 0.5f * (-phi_w9_f(dp) + phi_w9_f(dm));
            }
        };
        project(std::integral_constant<int, 0>{});
        project(std::integral_constant<int, 1>{});
        project(std::integral_constant<int, 2>{});
        project(std::integral_constant<int, 3>{});
        project(std::integral_constant<int, 4>{});

        auto assemble = [&](auto mm) {
            constexpr int m = decltype(mm)::value;
            const double *F = &sm[(V_F0 + m) * NW];
            double th;
            if constexpr (S == 5) {
                th = 1. / 12. * (-1. * (F[oc - 1] + F[oc + 2]) + 7. * (F[oc] + F[oc + 1]));
            } else {
                th = 1. / 840. * (533. * (F[oc + 1] + F[oc]) - 139. * (F[oc + 2] + F[oc - 1])
                                  + 29. * (F[oc + 3] + F[oc - 2]) - 3. * (F[oc + 4] + F[oc - 3]));
            }
            double Rr[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
            if constexpr (AX < 0) right_row<m>(e, Rr);
            else right_row_ax<m, (AX < 0 ? 0 : AX)>(e, nsig, Rr);
            float acc = 0.f;
#pragma unroll
            for (int cc = 0; cc < 5; cc++)
                if (AX < 0 || rnz(m, AX, cc)) acc += (float)Rr[cc] * phif[cc];
            out[m] = (double)acc + th;
        };
        assemble(std::integral_constant<int, 0>{});
        assemble(std::integral_constant<int, 1>{});
        assemble(std::integral_constant<int, 2>{});
        assemble(std::integral_constant<int, 3>{});
        assemble(std::integral_constant<int, 4>{});
    }
    double nxt[5];
    if constexpr (SHFL) {
#pragma unroll
        for (int m = 0; m < 5; m++) nxt[m] = next_lane(out[m]);
    } else {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 5; m++) sm[m * NT + t] = out[m];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 5; m++) nxt[m] = (di < TDI - 1) ? sm[m * NT + t + 1] : 0.0;
    }

    // phase 3: divergence into Q for the tile's TDI-1 nodes
    if (di < TDI - 1 && t < TA * TDI) {
        const int dn = d0 + di;
        const int pa = pa0 + ta;
        if (dn < a.nD && pa >= a.oA && pa < a.oA + a.nA) {
            const long n = bbase + (long)pa * a.sA + (long)(dn + a.oD) * a.sD;
#pragma unroll
            for (int m = 0; m < 5; m++) {
                double dv = nxt[m] - out[m];
                if constexpr (PAIRS) dv = dcur[m] + dv;
                if constexpr (KEEP) keep[m] = -dv;
                else a.q.f[m][n] = (a.first ? 0.0 : a.q.f[m][n]) - dv;
            }
        }
    }
}
// Waves per SIMD asked of the compiler: the diagonal FP64 W5 sweeps run four (122-128 VGPRs, at most two
// spilled), which the LDS of an 8 x 32 or 4 x 64 tile allows too; at three waves (132-134 VGPRs) the xi
// sweep took 0.87 ms at 256^3 against 0.83.  WENO9 and the general metric: three waves (138-168 VGPRs).
// The mixed form is left to the compiler.
template <int S, int AX, bool MIX>
constexpr int weno_min_waves() { return MIX ? 1 : (S == 5 && AX >= 0 ? 4 : 3); }

template <int S, int TA, int TDI, int AX, bool MIX>
__global__ __launch_bounds__(TA * TDI, (weno_min_waves<S, AX, MIX>())) void k_weno(WenoArgs a)
{
    __shared__ double lds[weno_lds<S, TA, TDI, AX, MIX>()];
    int bx, by, bz;
    sweep_tile(blockIdx.x, a.tg, bx, by, bz);
    weno_body<S, TA, TDI, AX, MIX>(a, bx, by, bz, lds);
}

// ---- viscous fluxes: face-based LDS sweep ------------------------------------------------
// CalcViscidFluxesIn{Xi,Eta,Zeta}DirectionDirectly (src/ZD.c:47-694) restructured by faces:
// the reference evaluates both half-point fluxes of every node; here each face flux of
// direction D is computed once from an LDS pencil and differenced.  Face values: midpoint
// derivatives of u,v,w,T along D and midpoint interpolations of the nodal cross derivatives;
// coefficients K = (mu fac)_face averages; energy work term u_i (F(i+1/2) - F(i-1/2)) and the
// nodal product term are evaluated per node as in the reference.
// Stage update of one interior node (src/Functions.c:2300-2365) with the manufactured source
// (Q += J src): shared by the last kernels of a stage, which apply it directly
// instead of storing Q.
struct RkArgs {
    CFields5 un, us, src;
    Fields5 out, qsum;
    double a, b, qf, ff, mf, tau;
    int first_stage, has_src, three;
    // end of step (the last stage of shx_run, shx_run_cfl and shx_simulate): checkNAN on the new
    // state and the CFL maximum over it, fused into the update.  nan_cnt: running count of
    // non-finite interior densities (those nodes get rho = u = v = w (= stored p) = 1e6);
    // cfl_red: the maximum of the node CFL sum, as the bits of a positive double
    int *nan_cnt;
    int *nan_flag;           // pinned host word set to 1 with the count, which the host reads after the
                             // step instead of copying the count (null in batches)
    gdp nanP;
    unsigned long long *cfl_red;
    double gamma, upsilon;
};

// Reductions over a wavefront (all 64 lanes active).
__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_sum(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// Maxima of non-negative doubles reduce into RED_SLOTS slots (positive doubles order like their
// bit patterns, so an unsigned 64-bit atomic max combines them); a block uses slot
// blockIdx % RED_SLOTS, and k_red_report takes the maximum of the slots.  One slot for a whole
// launch would serialise every wave's atomic on one cache line.
constexpr int RED_SLOTS = 256;
__device__ __forceinline__ void wave_max_to(unsigned long long *out, double v)
{
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0 && v > 0.0) {
        unsigned long long *slot = out + (blockIdx.x & (RED_SLOTS - 1));
        const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
        if (bits > *slot) atomicMax(slot, bits);     // a stale read only costs an extra atomic
    }
}

// CFL sum of one node, sum_d |theta_d| + c |grad xi_d| (the per-node spectral radius of
// src/WENO.c:1560-1615 with unit index spacing); m: the node's metric rows xi_x .. zeta_z.
// Shared by k_cfl_max and the fused end-of-step check, which therefore give the same bits.
// DIAG (the off-diagonal entries are zero): |grad xi_d| = |m_dd|, which is what the general form
// gives, since u m_dd + v 0 + w 0 = u m_dd and sqrt(m_dd^2 + 0 + 0) = |m_dd| exactly (a correctly
// rounded square root of a rounded square is the operand's magnitude).
template <bool DIAG = false>
__device__ __forceinline__ double node_cfl_sum(const double gamma, const double upsilon, const int dims,
                                               const double rho, const double u, const double v, const double w,
                                               const double e, const double m[9])
{
    const double p = fabs(rho * (gamma - 1) / upsilon * (e - 0.5 * ((u * u) + (v * v) + (w * w))));
    const double cs = sqrt(upsilon * gamma * p / rho);
    double s = 0.0;
    // unrolled over three directions with a guard, so that m and uu stay in registers
    if constexpr (DIAG) {
        const double uu[3] = {u, v, w};
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (d < dims) {
                const double a = m[4 * d];
                s += fabs(uu[d] * a) + cs * fabs(a);
            }
        }
    } else {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (d < dims) {
                const double a = m[3 * d], b = m[3 * d + 1], z = m[3 * d + 2];
                s += fabs(u * a + v * b + w * z) + cs * sqrt(a * a + b * b + z * z);
            }
        }
    }
    return s;
}

// The node's U_n and Q_sum loaded ahead of the update (rk_preload), so that a fused sweep can
// issue those loads before its window and flux work and their latency overlaps that work.
struct RkPre { double un[5], qs[5]; };
__device__ __forceinline__ void rk_preload(const RkArgs &A, const long n, RkPre &p)
{
#pragma unroll
    for (int m = 0; m < 5; m++) {
        p.un[m] = (m == 3 && !A.three) ? 0.0 : A.un.f[m][n];
        p.qs[m] = A.first_stage ? 0.0 : A.qsum.f[m][n];
    }
}

// m9, cfl: the node's metric rows and where its CFL sum goes (read only when A.cfl_red is set);
// DIAG: the metric is diagonal (node_cfl_sum); pre: U_n and Q_sum loaded by rk_preload
template <bool DIAG = false>
__device__ __forceinline__ void rk_point(const RkArgs &A, const long n, const double J, double qv[5],
                                         const double *m9 = nullptr, double *cfl = nullptr,
                                         const RkPre *pre = nullptr)
{
    if (A.has_src) {
        qv[0] += J * A.src.f[0][n];
        qv[1] += J * A.src.f[1][n];
        qv[2] += J * A.src.f[2][n];
        if (A.three) qv[3] += J * A.src.f[3][n];
        qv[4] += J * A.src.f[4][n];
    }
    double qs[5];
#pragma unroll
    for (int m = 0; m < 5; m++) {
        const double old = A.first_stage ? 0.0 : (pre ? pre->qs[m] : A.qsum.f[m][n]);
        qs[m] = old + A.mf * qv[m];
        if (A.mf != 0.0) A.qsum.f[m][n] = qs[m];
    }
    const double tj = A.tau / J;
    const double rho_n = pre ? pre->un[0] : A.un.f[0][n];
    // b = 0 on every RK4 stage and the first SSP-RK3 stage: U_s is not read there
    const double rho_s = (A.b != 0.0) ? A.us.f[0][n] : 0.0;
    const double rho = A.a * rho_n + A.b * rho_s + tj * (A.qf * qv[0] + A.ff * qs[0]);
    A.out.f[0][n] = rho;
    double nv[5];
    nv[0] = rho;
#pragma unroll
    for (int m = 1; m < 5; m++) {
        if (m == 3 && !A.three) { A.out.f[3][n] = 0.0; nv[3] = 0.0; continue; }
        const double us = (A.b != 0.0) ? A.us.f[m][n] : 0.0;
        nv[m] = (A.a * (pre ? pre->un[m] : A.un.f[m][n]) * rho_n + A.b * us * rho_s
                 + tj * (A.qf * qv[m] + A.ff * qs[m])) / rho;
        A.out.f[m][n] = nv[m];
    }
    if (A.nan_cnt && !isfinite(rho)) {
        // checkNAN (src/Functions.c:5419-5467) on the step's U_RK
        A.out.f[0][n] = 1000000; A.out.f[1][n] = 1000000; A.out.f[2][n] = 1000000; A.out.f[3][n] = 1000000;
        if (A.nanP) A.nanP[n] = 1000000;
        atomicAdd(A.nan_cnt, 1);
        if (A.nan_flag) __hip_atomic_store(A.nan_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    } else if (A.cfl_red && cfl) {
        *cfl = node_cfl_sum<DIAG>(A.gamma, A.upsilon, A.three ? 3 : 2, nv[0], nv[1], nv[2], nv[3], nv[4], m9);
    }
}

struct ViscArgs {
    gcdp u, v, w, T, mu;
    gcdp cr[8];                   // cross derivatives (layout depends on DIAG, see host)
    CFields10 met;
    Fields5 q;
    long sD, sA, sB;
    int nD, nA, nB, oD, oA, oB, ngD;
    int ngA;                      // padded extent of the A axis
    int coalesce_d;
    int alignA;
    int bug;                      // zeta stencil k offset taken from j (DIR = 2 only)
    int fuse_rk;                  // last sweep of the stage: apply the stage update (rk)
    int iso_hi;                   // the upper face of the sweep direction is an isothermal wall:
    double gam_iso;               // the last interior node's heat-conduction factor (the mean of
                                  // its own and the wall ghost's, src/ZD.c:193-194)
    int tg[4];                    // tile grid and order of a single-case launch
    RkArgs rk;
    Consts k;
};

template <int DIR> struct Others { static constexpr int b1 = (DIR == 0) ? 1 : 0; static constexpr int b2 = (DIR == 2) ? 1 : 2; };

// Viscous flux of one node's metric along row a = DIR, without J and mu: the reference's factors
// fac_{i,k,b} (CreateViscidMetric, src/Functions.c:6245-6386) contracted with the slot values d (velocity
// derivative d[3k+b], T at 9+b).  fac is the Newtonian stress in metric rows, so the sum over k and b is the
// stress of the Cartesian velocity gradient g_kj = sum_b d_kb r_bj along a:
//   t_i = sum_j (g_ij + g_ji) a_j - 2/3 a_i div g,   t_3 = grad T . a.
// 57 operations where evaluating the 30 factors takes 180.
template <int DIR>
__device__ __forceinline__ void stress_along(const double d[12], const double m[10], double t[4])
{
    double g[3][3];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < 3; j++) g[k][j] = d[3 * k] * m[j] + d[3 * k + 1] * m[3 + j] + d[3 * k + 2] * m[6 + j];
    const double *a = m + 3 * DIR;
    const double div = g[0][0] + g[1][1] + g[2][2];
    const double p = (2. / 3.) * div;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double acc = -(p * a[i]);
#pragma unroll
        for (int j = 0; j < 3; j++) acc += (g[i][j] + g[j][i]) * a[j];
        t[i] = acc;
    }
    t[3] = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) t[3] += (d[9] * m[j] + d[10] * m[3 + j] + d[11] * m[6 + j]) * a[j];
}
// face flux (momentum x,y,z and heat): the reference's mean of mu fac over the face's two nodes
template <int DIR>
__device__ __forceinline__ void face_flux_generic(const double d[12], const double m0[10], const double m1[10],
                                                  const double mu0, const double mu1, double F[4])
{
    double t0[4], t1[4];
    stress_along<DIR>(d, m0, t0);
    stress_along<DIR>(d, m1, t1);
    const double w0 = 0.5 * (mu0 * m0[9]), w1 = 0.5 * (mu1 * m1[9]);
#pragma unroll
    for (int i = 0; i < 4; i++) F[i] = w0 * t0[i] + w1 * t1[i];
}

// diagonal metric (the reference's 3D metric): node values mD (row D, component D), mb[3]
// (diagonal entries of all rows), J.  Only the non-zero factors of the generic table remain.
template <int DIR>
__device__ __forceinline__ void face_flux_diag(const double d[12], const double g0[3], const double J0,
                                               const double g1[3], const double J1, const double mu0,
                                               const double mu1, double F[4])
{
    const double mD0 = g0[DIR], mD1 = g1[DIR];
    const double KA = 0.5 * (mu0 * (J0 * (mD0 * mD0)) + mu1 * (J1 * (mD1 * mD1)));
    const double K43 = 0.5 * (mu0 * (J0 * (4.0 / 3.0 * mD0 * mD0)) + mu1 * (J1 * (4.0 / 3.0 * mD1 * mD1)));
    double FD = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (k == DIR) { FD += d[k * 3 + k] * K43; continue; }
        const double KC = 0.5 * (mu0 * (J0 * (-2.0 / 3.0 * g0[k] * mD0)) + mu1 * (J1 * (-2.0 / 3.0 * g1[k] * mD1)));
        FD += d[k * 3 + k] * KC;
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        if (i == DIR) { F[i] = FD; continue; }
        const double KB = 0.5 * (mu0 * (J0 * (g0[i] * mD0)) + mu1 * (J1 * (g1[i] * mD1)));
        F[i] = d[DIR * 3 + i] * KB + d[i * 3 + DIR] * KA;
    }
    F[3] = d[9 + DIR] * KA;
}

// nodal product term sum_blk g_{blk,D} sum_s g_s mu fac_{blk,s} (src/ZD.c:230-266); g: nodal velocity
// derivatives (slots as above)
template <int DIR>
__device__ __forceinline__ double node_prod_generic(const double g[12], const double m[10], const double mu)
{
    double t[4];
    stress_along<DIR>(g, m, t);
    return (mu * m[9]) * (g[DIR] * t[0] + g[3 + DIR] * t[1] + g[6 + DIR] * t[2]);
}

template <int DIR>
__device__ __forceinline__ double node_prod_diag(const double g[9], const double gm[3], const double J, const double mu)
{
    const double mD = gm[DIR];
    double prod = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double gd = g[i * 3 + DIR];
        if (i == DIR) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double f = (k == DIR) ? J * (4.0 / 3.0 * mD * mD) : J * (-2.0 / 3.0 * gm[k] * mD);
                prod += gd * g[k * 3 + k] * mu * f;
            }
        } else {
            prod += gd * g[DIR * 3 + i] * mu * (J * (gm[i] * mD));
            prod += gd * g[i * 3 + DIR] * mu * (J * (mD * mD));
        }
    }
    return prod;
}

// LDS slots
enum { VS_U, VS_V, VS_W, VS_T, VS_MU, VS_CR };

// LDS of one viscous sweep block, in doubles: the node window (diagonal metric: 13 fields; general: 12
// fields, and in their place, once the face's and node's derivatives are in registers, mu and the metric
// of the tile's nodes and the one below them), and the zeta-index quirk's line values.  Plus-side face
// values go from each thread to the previous one by a lane move (the minus side stays in registers): a
// tile row never straddles two wavefronts.
template <int S, int DIR, int TA, int TDI, bool DIAG>
constexpr int visc_lds()
{
    constexpr int G = (S + 1) / 2, NW = (TDI - 1 + 2 * G) * TA;
    constexpr int NC = DIAG ? 4 : 8, NLV = 4 + NC, NP = 2 * G + 1;
    constexpr int WIN = DIAG ? (VS_CR + NC + 4) * NW : std::max((4 + NC) * NW, 11 * (TDI + 1) * TA);
    static_assert(64 % TDI == 0, "tile rows stay in one wavefront");
    return WIN + ((DIR == 2) ? TA * NP * NLV + TA * 2 * NLV : 0);
}

// ADD: add add[5] (a fused WENO sweep's contribution of the thread's node) to Q before the
// viscous terms.  PRE: load the node's Q (and U_n, Q_sum for the stage update) before the window.
template <int S, int DIR, int TA, int TDI, bool ADD = false, bool PRE = false>
__device__ __forceinline__ void visc_diag_body(const ViscArgs &a, const int bx, const int by, const int bz,
                                          double *lds, const double *add = nullptr)
{
    constexpr int G = (S + 1) / 2;
    constexpr int WD = TDI - 1 + 2 * G;
    constexpr int NW = WD * TA;
    constexpr int NT = TA * TDI;
    constexpr int NC = 4;                            // cross-derivative fields
    constexpr int NM = 4;                            // metric values per node
    constexpr int VS_M = VS_CR + NC;
    constexpr int NVS = VS_M + NM;
    constexpr int b1 = Others<DIR>::b1, b2 = Others<DIR>::b2;
    constexpr int NP = 2 * G + 1;                    // line positions used by the zeta-index quirk
    constexpr int NLV = 4 + NC;                      // values per position: u,v,w,T + cross
    double *const sm = lds;
    double *const line = sm + NVS * NW;
    double *const lined = line + TA * NP * NLV;

    const int t = threadIdx.x;
    // first padded A index of the tile (aligned to TA when the A axis is contiguous in memory)
    const int pa0 = a.alignA ? bx * TA : bx * TA + a.oA;
    const int b = by;
    const int d0 = bz * (TDI - 1);
    const long bbase = (long)(b + a.oB) * a.sB;
    const Consts &k = a.k;
    const int ta = t / TDI, di = t - ta * TDI;
    const int dn = d0 + di, pa = pa0 + ta;
    const bool own = di < TDI - 1 && dn < a.nD && pa >= a.oA && pa < a.oA + a.nA;
    const long n = bbase + (long)pa * a.sA + (long)(dn + a.oD) * a.sD;
    // PRE: the node's Q, and U_n and Q_sum where the sweep applies the stage update, are loaded
    // before the window, so that their latency overlaps the staging and the face fluxes
    double q0[5];
    RkPre pre;
    if (PRE && own) {
#pragma unroll
        for (int m = 0; m < 5; m++) q0[m] = a.q.f[m][n];
        if (a.fuse_rk) rk_preload(a.rk, n, pre);
    }

    for (int idx = t; idx < NW; idx += NT) {
        int aa, dd;
        if (a.coalesce_d) { aa = idx / WD; dd = idx - aa * WD; }
        else { dd = idx / TA; aa = idx - dd * TA; }
        const int pa = max(a.oA, min(pa0 + aa, a.oA + a.nA - 1));
        int dp = d0 - G + dd + a.oD;
        dp = max(0, min(dp, a.ngD - 1));
        const long n = bbase + (long)pa * a.sA + (long)dp * a.sD;
        const int o = aa * WD + dd;
        sm[VS_U * NW + o] = a.u[n];
        sm[VS_V * NW + o] = a.v[n];
        sm[VS_W * NW + o] = a.w[n];
        sm[VS_T * NW + o] = a.T[n];
        sm[VS_MU * NW + o] = a.mu[n];
#pragma unroll
        for (int c = 0; c < NC; c++) sm[(VS_CR + c) * NW + o] = a.cr[c][n];
        sm[(VS_M + 0) * NW + o] = a.met.f[0][n];
        sm[(VS_M + 1) * NW + o] = a.met.f[4][n];
        sm[(VS_M + 2) * NW + o] = a.met.f[8][n];
        sm[(VS_M + 3) * NW + o] = a.met.f[9][n];
    }
    const bool bug = (DIR == 2) && a.bug;
    if (bug) {
        // the reference's zeta stencil (src/ZD.c:547-548) reads positions k' = j + l - g on the
        // (i, j) line for every k: the face values are constant along the line
        for (int idx = t; idx < TA * NP * NLV; idx += NT) {
            const int ln = idx / (NP * NLV);
            const int rem = idx - ln * NP * NLV;
            const int pos = rem / NLV, f = rem - pos * NLV;
            const int jpad = max(a.oA, min(pa0 + ln, a.oA + a.nA - 1));   // A axis is j for DIR = 2
            // the reference's index (i ng_j + j) ng_k + k' with k' = j - g + pos in its unpadded
            // k-fastest layout: where k' passes the row end (ng_j > ng_k) it reads the next rows
            // (or the next plane's first ones), which the padded layout finds at (j', k'') below
            const int kq = jpad - G + pos;
            long n;
            if (kq < a.ngD) {
                n = bbase + (long)jpad * a.sA + kq;
            } else {
                int jr = jpad + kq / a.ngD;
                const int kr = kq % a.ngD;
                const int ia = jr / a.ngA;
                jr -= ia * a.ngA;
                n = bbase + (long)ia * a.sB + (long)jr * a.sA + kr;
            }
            double val;
            if (f == 0) val = a.u[n];
            else if (f == 1) val = a.v[n];
            else if (f == 2) val = a.w[n];
            else if (f == 3) val = a.T[n];
            else val = a.cr[f - 4][n];
            line[(ln * NP + pos) * NLV + f] = val;
        }
    }
    __syncthreads();
    if (bug && di < 2) {
        // di = 0: minus-side values (positions 0..S), di = 1: plus side (positions 1..S+1)
        const double *Lp = &line[(ta * NP + di) * NLV];
#pragma unroll
        for (int f = 0; f < NLV; f++) {
            double acc = 0.0;
            const double *cf = (f < 4) ? k.zd_mid : k.zd_int;
#pragma unroll
            for (int l = 0; l <= S; l++) acc += cf[l] * Lp[l * NLV + f];
            lined[(ta * 2 + di) * NLV + f] = acc;
        }
    }
    if (bug) __syncthreads();

    const int ob = ta * WD + di;
    const int oc = ob + G - 1;
    double out[8];
    {
        const double mu0 = sm[VS_MU * NW + oc], mu1 = sm[VS_MU * NW + oc + 1];
        // slot layout d[k*3+b], T at 9+b
        auto face = [&](const double *own4, const double *cr, double F[4]) {
            double d[12];
#pragma unroll
            for (int s = 0; s < 12; s++) d[s] = 0.0;
            d[0 * 3 + DIR] = own4[0]; d[1 * 3 + DIR] = own4[1]; d[2 * 3 + DIR] = own4[2]; d[9 + DIR] = own4[3];
            d[b1 * 3 + b1] = cr[0]; d[DIR * 3 + b1] = cr[1];
            d[b2 * 3 + b2] = cr[2]; d[DIR * 3 + b2] = cr[3];
            double g0[3], g1[3];
            g0[0] = sm[(VS_M + 0) * NW + oc]; g0[1] = sm[(VS_M + 1) * NW + oc]; g0[2] = sm[(VS_M + 2) * NW + oc];
            g1[0] = sm[(VS_M + 0) * NW + oc + 1]; g1[1] = sm[(VS_M + 1) * NW + oc + 1]; g1[2] = sm[(VS_M + 2) * NW + oc + 1];
            face_flux_diag<DIR>(d, g0, sm[(VS_M + 3) * NW + oc], g1, sm[(VS_M + 3) * NW + oc + 1], mu0, mu1, F);
        };
        if (!bug) {
            double own4[4] = {0.0, 0.0, 0.0, 0.0}, cr[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) cr[c] = 0.0;
#pragma unroll
            for (int l = 0; l <= S; l++) {
                const double cm = k.zd_mid[l], ci = k.zd_int[l];
                own4[0] += cm * sm[VS_U * NW + ob + l];
                own4[1] += cm * sm[VS_V * NW + ob + l];
                own4[2] += cm * sm[VS_W * NW + ob + l];
                own4[3] += cm * sm[VS_T * NW + ob + l];
#pragma unroll
                for (int c = 0; c < NC; c++) cr[c] += ci * sm[(VS_CR + c) * NW + ob + l];
            }
            double F[4];
            face(own4, cr, F);
#pragma unroll
            for (int m = 0; m < 4; m++) { out[m] = F[m]; out[4 + m] = F[m]; }
        } else {
            double FA[4], FB[4];
            face(&lined[(ta * 2 + 0) * NLV], &lined[(ta * 2 + 0) * NLV + 4], FA);
            face(&lined[(ta * 2 + 1) * NLV], &lined[(ta * 2 + 1) * NLV + 4], FB);
#pragma unroll
            for (int m = 0; m < 4; m++) { out[m] = FA[m]; out[4 + m] = FB[m]; }
        }
    }
    double nxt[4];
#pragma unroll
    for (int m = 0; m < 4; m++) nxt[m] = next_lane(out[4 + m]);

    double cflv = 0.0;                           // CFL sum of this thread's node (end-of-step check)
    if (di < TDI - 1) {
        if (own) {
            const int p = ob + G;                    // window position of this node
            // faces: minus = this thread's face (A values), plus = next thread's face (B values)
            double dF[4];
#pragma unroll
            for (int m = 0; m < 4; m++) dF[m] = nxt[m] - out[m];
            // nodal gradients: own-direction derivatives from the window, cross ones stored
            double g[9];
#pragma unroll
            for (int s = 0; s < 9; s++) g[s] = 0.0;
            {
                double du = 0.0, dv = 0.0, dw = 0.0;
#pragma unroll
                for (int l = 0; l <= S + 1; l++) {
                    du += k.zd_der[l] * sm[VS_U * NW + ob + l];
                    dv += k.zd_der[l] * sm[VS_V * NW + ob + l];
                    dw += k.zd_der[l] * sm[VS_W * NW + ob + l];
                }
                g[0 * 3 + DIR] = du; g[1 * 3 + DIR] = dv; g[2 * 3 + DIR] = dw;
            }
            const double mu = sm[VS_MU * NW + p];
            g[b1 * 3 + b1] = sm[(VS_CR + 0) * NW + p]; g[DIR * 3 + b1] = sm[(VS_CR + 1) * NW + p];
            g[b2 * 3 + b2] = sm[(VS_CR + 2) * NW + p]; g[DIR * 3 + b2] = sm[(VS_CR + 3) * NW + p];
            const double gmv[3] = {sm[(VS_M + 0) * NW + p], sm[(VS_M + 1) * NW + p], sm[(VS_M + 2) * NW + p]};
            const double prod = node_prod_diag<DIR>(g, gmv, sm[(VS_M + 3) * NW + p], mu);
            const double work = sm[VS_U * NW + p] * dF[0] + sm[VS_V * NW + p] * dF[1] + sm[VS_W * NW + p] * dF[2];
#pragma unroll
            for (int m = 0; m < 5; m++) {
                const double qn = PRE ? q0[m] : a.q.f[m][n];
                q0[m] = ADD ? qn + add[m] : qn;
            }
            if (a.fuse_rk) {
                double qv[5];
                qv[0] = q0[0];
                qv[1] = q0[1] + k.psi * dF[0];
                qv[2] = q0[2] + k.psi * dF[1];
                qv[3] = q0[3] + k.psi * dF[2];
                const double gh = (a.iso_hi && dn == a.nD - 1) ? a.gam_iso : k.gam_heat;
                qv[4] = q0[4] + (gh * dF[3] + k.psi * (work + prod));
                const double J = sm[(VS_M + 3) * NW + p];
                if (a.rk.cfl_red) {
                    // end of step: the node's metric rows for its CFL sum
                    double m9[9];
#pragma unroll
                    for (int c = 0; c < 9; c++) m9[c] = 0.0;
                    m9[0] = sm[(VS_M + 0) * NW + p]; m9[4] = sm[(VS_M + 1) * NW + p]; m9[8] = sm[(VS_M + 2) * NW + p];
                    rk_point<true>(a.rk, n, J, qv, m9, &cflv, PRE ? &pre : nullptr);
                } else {
                    rk_point(a.rk, n, J, qv, nullptr, nullptr, PRE ? &pre : nullptr);
                }
            } else {
                if (ADD) a.q.f[0][n] = q0[0];
                a.q.f[1][n] = q0[1] + k.psi * dF[0];
                a.q.f[2][n] = q0[2] + k.psi * dF[1];
                a.q.f[3][n] = q0[3] + k.psi * dF[2];
                const double gh = (a.iso_hi && dn == a.nD - 1) ? a.gam_iso : k.gam_heat;
                a.q.f[4][n] = q0[4] + (gh * dF[3] + k.psi * (work + prod));
            }
        }
    }
    if (a.rk.cfl_red) wave_max_to(a.rk.cfl_red, cflv);
}
// General metric.  The window holds the differentiated fields only (u, v, w, T and eight cross
// derivatives); once every thread has its face's derivatives and its node's, mu and the metric of the
// tile's nodes take its place.  Bound by latency: with the metric in the window the 16 x 12 tile needed
// 56 KB and 168 VGPRs, six waves per CU; with it, and the 30 factors per face in place of the stress
// contraction, 119 x 96 x 104 took 128, 113 and 172 us along xi, eta and zeta (with the update), 78, 75 and
// 123 now.
template <int S, int DIR, int TA, int TDI>
__device__ __forceinline__ void visc_gen_body(const ViscArgs &a, const int bx, const int by, const int bz, double *lds)
{
    constexpr int G = (S + 1) / 2;
    constexpr int WD = TDI - 1 + 2 * G;
    constexpr int NW = WD * TA;
    constexpr int NT = TA * TDI;
    constexpr int NC = 8;                            // cross-derivative fields
    constexpr int b1 = Others<DIR>::b1, b2 = Others<DIR>::b2;
    constexpr int NP = 2 * G + 1;                    // line positions used by the zeta-index quirk
    constexpr int NLV = 4 + NC;                      // values per position: u,v,w,T + cross
    constexpr int MD = TDI + 1, NM = MD * TA;        // metric window: the nodes of a row's faces
    double *const sm = lds;
    double *const line = sm + (NLV * NW > 11 * NM ? NLV * NW : 11 * NM);
    double *const lined = line + TA * NP * NLV;

    const int t = threadIdx.x;
    const int pa0 = a.alignA ? bx * TA : bx * TA + a.oA;
    const int b = by;
    const int d0 = bz * (TDI - 1);
    const long bbase = (long)(b + a.oB) * a.sB;
    const Consts &k = a.k;
    const int ta = t / TDI, di = t - ta * TDI;
    const int dn = d0 + di, pa = pa0 + ta;
    const bool own = di < TDI - 1 && dn < a.nD && pa >= a.oA && pa < a.oA + a.nA;
    const long n = bbase + (long)pa * a.sA + (long)(dn + a.oD) * a.sD;

    for (int idx = t; idx < NW; idx += NT) {
        int aa, dd;
        if (a.coalesce_d) { aa = idx / WD; dd = idx - aa * WD; }
        else { dd = idx / TA; aa = idx - dd * TA; }
        const int pa = max(a.oA, min(pa0 + aa, a.oA + a.nA - 1));
        int dp = d0 - G + dd + a.oD;
        dp = max(0, min(dp, a.ngD - 1));
        const long n = bbase + (long)pa * a.sA + (long)dp * a.sD;
        const int o = aa * WD + dd;
        sm[0 * NW + o] = a.u[n];
        sm[1 * NW + o] = a.v[n];
        sm[2 * NW + o] = a.w[n];
        sm[3 * NW + o] = a.T[n];
#pragma unroll
        for (int c = 0; c < NC; c++) sm[(4 + c) * NW + o] = a.cr[c][n];
    }
    const bool bug = (DIR == 2) && a.bug;
    if (bug) {
        // the reference's zeta stencil (src/ZD.c:547-548) reads positions k' = j + l - g on the
        // (i, j) line for every k: the face values are constant along the line
        for (int idx = t; idx < TA * NP * NLV; idx += NT) {
            const int ln = idx / (NP * NLV);
            const int rem = idx - ln * NP * NLV;
            const int pos = rem / NLV, f = rem - pos * NLV;
            const int jpad = max(a.oA, min(pa0 + ln, a.oA + a.nA - 1));   // A axis is j for DIR = 2
            // the reference's index (i ng_j + j) ng_k + k' with k' = j - g + pos in its unpadded
            // k-fastest layout: where k' passes the row end (ng_j > ng_k) it reads the next rows
            // (or the next plane's first ones), which the padded layout finds at (j', k'') below
            const int kq = jpad - G + pos;
            long n;
            if (kq < a.ngD) {
                n = bbase + (long)jpad * a.sA + kq;
            } else {
                int jr = jpad + kq / a.ngD;
                const int kr = kq % a.ngD;
                const int ia = jr / a.ngA;
                jr -= ia * a.ngA;
                n = bbase + (long)ia * a.sB + (long)jr * a.sA + kr;
            }
            double val;
            if (f == 0) val = a.u[n];
            else if (f == 1) val = a.v[n];
            else if (f == 2) val = a.w[n];
            else if (f == 3) val = a.T[n];
            else val = a.cr[f - 4][n];
            line[(ln * NP + pos) * NLV + f] = val;
        }
    }
    __syncthreads();
    if (bug && di < 2) {
        // di = 0: minus-side values (positions 0..S), di = 1: plus side (positions 1..S+1)
        const double *Lp = &line[(ta * NP + di) * NLV];
#pragma unroll
        for (int f = 0; f < NLV; f++) {
            double acc = 0.0;
            const double *cf = (f < 4) ? k.zd_mid : k.zd_int;
#pragma unroll
            for (int l = 0; l <= S; l++) acc += cf[l] * Lp[l * NLV + f];
            lined[(ta * 2 + di) * NLV + f] = acc;
        }
    }
    if (bug) __syncthreads();

    const int ob = ta * WD + di;
    double fv[NLV];                                  // the face's derivatives (own u,v,w,T; cross)
    double dv[3] = {0.0, 0.0, 0.0}, vel[3], gc[6];   // the node's: along the direction, velocity, cross
#pragma unroll
    for (int f = 0; f < NLV; f++) fv[f] = 0.0;
    if (!bug) {
#pragma unroll
        for (int l = 0; l <= S; l++) {
            const double cm = k.zd_mid[l], ci = k.zd_int[l];
#pragma unroll
            for (int f = 0; f < NLV; f++) fv[f] += (f < 4 ? cm : ci) * sm[f * NW + ob + l];
        }
    }
#pragma unroll
    for (int l = 0; l <= S + 1; l++)
#pragma unroll
        for (int q = 0; q < 3; q++) dv[q] += k.zd_der[l] * sm[q * NW + ob + l];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        vel[q] = sm[q * NW + ob + G];
        gc[q] = sm[(4 + q) * NW + ob + G];
        gc[3 + q] = sm[(8 + q) * NW + ob + G];
    }
    __syncthreads();
    // mu and the metric, position dd of a row: node d0 - 1 + dd
    for (int idx = t; idx < NM; idx += NT) {
        int aa, dd;
        if (a.coalesce_d) { aa = idx / MD; dd = idx - aa * MD; }
        else { dd = idx / TA; aa = idx - dd * TA; }
        const int pa = max(a.oA, min(pa0 + aa, a.oA + a.nA - 1));
        const int dp = min(d0 - 1 + dd + a.oD, a.ngD - 1);
        const long n = bbase + (long)pa * a.sA + (long)dp * a.sD;
        const int o = aa * MD + dd;
#pragma unroll
        for (int c = 0; c < 10; c++) sm[c * NM + o] = a.met.f[c][n];
        sm[10 * NM + o] = a.mu[n];
    }
    __syncthreads();
    const int mo = ta * MD + di;                     // the face's lower node; the thread's node is the next
    double m1[10];
#pragma unroll
    for (int c = 0; c < 10; c++) m1[c] = sm[c * NM + mo + 1];
    const double mu1 = sm[10 * NM + mo + 1];
    double F[4], nxt[4];
    {
        double m0[10];
#pragma unroll
        for (int c = 0; c < 10; c++) m0[c] = sm[c * NM + mo];
        const double mu0 = sm[10 * NM + mo];
        // slot layout d[k*3+b], T at 9+b
        auto face = [&](const double *v, double *F) {
            double d[12];
#pragma unroll
            for (int q = 0; q < 4; q++) { d[3 * q + DIR] = v[q]; d[3 * q + b1] = v[4 + q]; d[3 * q + b2] = v[8 + q]; }
            face_flux_generic<DIR>(d, m0, m1, mu0, mu1, F);
        };
        if (!bug) {
            face(fv, F);
#pragma unroll
            for (int q = 0; q < 4; q++) nxt[q] = F[q];
        } else {
            face(&lined[(ta * 2 + 0) * NLV], F);
            face(&lined[(ta * 2 + 1) * NLV], nxt);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) nxt[q] = next_lane(nxt[q]);

    double cflv = 0.0;                               // CFL sum of this thread's node (end-of-step check)
    if (own) {
        double dF[4], g[12];
#pragma unroll
        for (int q = 0; q < 4; q++) dF[q] = nxt[q] - F[q];
#pragma unroll
        for (int q = 0; q < 3; q++) { g[3 * q + DIR] = dv[q]; g[3 * q + b1] = gc[q]; g[3 * q + b2] = gc[3 + q]; g[9 + q] = 0.0; }
        const double prod = node_prod_generic<DIR>(g, m1, mu1);
        const double work = vel[0] * dF[0] + vel[1] * dF[1] + vel[2] * dF[2];
        const double gh = (a.iso_hi && dn == a.nD - 1) ? a.gam_iso : k.gam_heat;
        double qv[5];
#pragma unroll
        for (int q = 0; q < 5; q++) qv[q] = a.q.f[q][n];
#pragma unroll
        for (int q = 0; q < 3; q++) qv[1 + q] = qv[1 + q] + k.psi * dF[q];
        qv[4] = qv[4] + (gh * dF[3] + k.psi * (work + prod));
        if (a.fuse_rk) {
            rk_point(a.rk, n, m1[9], qv, m1, &cflv);
        } else {
#pragma unroll
            for (int q = 1; q < 5; q++) a.q.f[q][n] = qv[q];
        }
    }
    if (a.rk.cfl_red) wave_max_to(a.rk.cfl_red, cflv);
}
template <int S, int DIR, int TA, int TDI, bool DIAG>
__device__ __forceinline__ void visc_body(const ViscArgs &a, const int bx, const int by, const int bz, double *lds)
{
    if constexpr (DIAG) visc_diag_body<S, DIR, TA, TDI>(a, bx, by, bz, lds);
    else visc_gen_body<S, DIR, TA, TDI>(a, bx, by, bz, lds);
}
template <int S, int DIR, int TA, int TDI, bool DIAG>
__global__ __launch_bounds__(TA * TDI) void k_visc_sweep(ViscArgs a)
{
    __shared__ double lds[visc_lds<S, DIR, TA, TDI, DIAG>()];
    int bx, by, bz;
    sweep_tile(blockIdx.x, a.tg, bx, by, bz);
    visc_body<S, DIR, TA, TDI, DIAG>(a, bx, by, bz, lds);
}

// ---- fused zeta direction: WENO and viscous sweeps and the stage update ----------------------
// One block sweeps a 4 x 64 tile (or 8 x 32, zeta_tile) along zeta twice.  The WENO phase keeps each node's inviscid
// divergence in registers; after a barrier the viscous phase reloads its window into the same LDS,
// adds that divergence and its own terms to Q and applies the stage update (or stores Q).  Q of
// this direction is read once instead of read-written by two kernels, and blocks in their WENO
// phase (VALU-bound) overlap blocks in their viscous phase (memory-bound).  Used for 3D cases with
// the diagonal metric, viscous runs only.
struct ZetaArgs { WenoArgs w; ViscArgs v; };
template <int S, int TA, int TDI, bool MIX>
constexpr int zeta_lds()
{
    return std::max(weno_lds<S, TA, TDI, 2, MIX>(), visc_lds<S, 2, TA, TDI, true>());
}
template <int S, int TA, int TDI, bool MIX>
__device__ __forceinline__ void zeta_body(const ZetaArgs &z, const int bx, const int by, const int bz, double *lds)
{
    double inv[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    weno_body<S, TA, TDI, 2, MIX, true>(z.w, bx, by, bz, lds, inv);
    __syncthreads();
    // Q, U_n and Q_sum loaded ahead (measured at 256^3: 1.95 -> 1.75 ms; the same in the fused eta
    // kernel, which stores Q instead of updating the stage, made it slower)
    visc_diag_body<S, 2, TA, TDI, true, true>(z.v, bx, by, bz, lds, inv);
}
// FP64 W5: held to 128 VGPRs (four waves per SIMD, as the LDS allows): 1.55 ms at 256^3 against
// 1.67 at three waves
template <int S, int TA, int TDI, bool MIX>
__global__ __launch_bounds__(TA * TDI, (weno_min_waves<S, 2, MIX>())) void k_zeta(ZetaArgs z)
{
    __shared__ double lds[zeta_lds<S, TA, TDI, MIX>()];
    int bx, by, bz;
    sweep_tile(blockIdx.x, z.w.tg, bx, by, bz);
    zeta_body<S, TA, TDI, MIX>(z, bx, by, bz, lds);
}

// ---- fused eta direction: WENO and viscous eta sweeps in one kernel ----------------------------
// One block sweeps an 8 x 32 tile along eta twice, as the fused zeta kernel does along zeta: the
// WENO phase keeps each node's inviscid divergence in registers, the viscous phase (after a barrier,
// in the same LDS) adds it and its own terms to Q, which this direction reads and writes once.
// 3D diagonal-metric viscous WENO5 cases, where the viscous xi terms ride on the derivative march.
struct EtaArgs { WenoArgs w; ViscArgs v; };
template <bool MIX>
constexpr int eta_lds()
{
    return weno_lds<5, 8, 32, 1, MIX>() > visc_lds<5, 1, 8, 32, true>() ? weno_lds<5, 8, 32, 1, MIX>()
                                                                       : visc_lds<5, 1, 8, 32, true>();
}
template <bool MIX>
__device__ __forceinline__ void eta_body(const EtaArgs &z, const int bx, const int by, const int bz, double *lds)
{
    double inv[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    weno_body<5, 8, 32, 1, MIX, true>(z.w, bx, by, bz, lds, inv);
    __syncthreads();
    visc_diag_body<5, 1, 8, 32, true>(z.v, bx, by, bz, lds, inv);
}
// FP64: four waves per SIMD (126 VGPRs; weno_flux)
constexpr int ETA_WAVES = 4;
template <bool MIX>
__global__ __launch_bounds__(256, (MIX ? 1 : ETA_WAVES)) void k_eta(EtaArgs z)
{
    __shared__ double lds[eta_lds<MIX>()];
    int bx, by, bz;
    sweep_tile(blockIdx.x, z.w.tg, bx, by, bz);
    eta_body<MIX>(z, bx, by, bz, lds);
}

// ---- WENO sweep along the contiguous axis (the last of the three) ------------------------------
// The inviscid stage's last kernel: the sweep keeps its node's divergence in registers, adds it to Q and
// applies the stage update (or stores Q, where viscous sweeps follow), instead of a separate pass that
// read Q back: 128 x 128 x 144 inviscid, sweep and update 138 + 100 us -> 188.
struct WenoLastArgs {
    WenoArgs w;
    CFields10 met;        // J, and the rows for the CFL sum of the end-of-step check
    int update;
    RkArgs rk;
};
template <int S, int TA, int TDI, int AX, bool MIX>
__device__ __forceinline__ void weno_last_body(const WenoLastArgs &z, const int bx, const int by, const int bz, double *lds)
{
    double keep[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, cfl = 0.0;
    weno_body<S, TA, TDI, AX, MIX, true>(z.w, bx, by, bz, lds, keep);
    const WenoArgs &a = z.w;
    const int ta = threadIdx.x / TDI, di = threadIdx.x % TDI;
    const int dn = bz * (TDI - 1) + di, pa = (a.alignA ? bx * TA : bx * TA + a.oA) + ta;
    if (di < TDI - 1 && dn < a.nD && pa >= a.oA && pa < a.oA + a.nA) {
        const long n = (long)(by + a.oB) * a.sB + (long)pa * a.sA + (long)(dn + a.oD) * a.sD;
        double q[5];
#pragma unroll
        for (int m = 0; m < 5; m++) q[m] = (a.first ? 0.0 : a.q.f[m][n]) + keep[m];
        if (z.update) {
            double m9[9];
#pragma unroll
            for (int c = 0; c < 9; c++) m9[c] = (z.rk.cfl_red && (AX < 0 || c % 4 == 0)) ? z.met.f[c][n] : 0.0;
            rk_point<(AX >= 0)>(z.rk, n, z.met.f[9][n], q, m9, &cfl);
        } else {
#pragma unroll
            for (int m = 0; m < 5; m++) a.q.f[m][n] = q[m];
        }
    }
    if (z.update && z.rk.cfl_red) wave_max_to(z.rk.cfl_red, cfl);
}
template <int S, int TA, int TDI, int AX, bool MIX>
__global__ __launch_bounds__(TA * TDI, (weno_min_waves<S, AX, MIX>())) void k_weno_last(WenoLastArgs z)
{
    __shared__ double lds[weno_lds<S, TA, TDI, AX, MIX>()];
    int bx, by, bz;
    sweep_tile(blockIdx.x, z.w.tg, bx, by, bz);
    weno_last_body<S, TA, TDI, AX, MIX>(z, bx, by, bz, lds);
}

// ---- viscous derivatives ------------------------------------------------------------------
// grad order: u_xi,u_eta,u_zeta, v_xi,v_eta,v_zeta, w_xi,w_eta,w_zeta, T_xi,T_eta,T_zeta.
// Direction d is evaluated where the node's d index is interior (all transverse nodes).
// 3D nodal derivatives, marching along i.  A block owns a GK x GJ column of (j, k) nodes over the
// full padded extent and walks a chunk of i planes: every plane is read from HBM once per chunk
// into LDS with a g-wide halo; the j and k derivatives come from there, the i derivative from a
// register window of 2g+1 plane centres per thread.  The T
// derivatives only when `tgrad` (the diagonal-metric viscous sweeps never read them).
//
// VX (3D diagonal metric): the viscous xi direction rides along (CalcViscidFluxesInXiDirection-
// Directly, src/ZD.c:47-260).  The march already holds, per column, the u, v, w window along i and
// each plane's eta and zeta derivatives; with T, mu and the metric of the column read as the planes
// pass, face i+1/2 follows at plane i+g from rings of the last 2g planes, and node i adds its xi
// viscous terms to Q.  The face and node arithmetic is the xi sweep's (k_visc_sweep<..,0,..>) term
// for term, so Q gets the same bits; u_eta and u_zeta, which only the xi direction reads, are not
// stored.
constexpr int GK = 64, GJ = 16;
struct GradArgs {
    CFields5 pr;
    gcdp T;
    Fields12 gr;
    Geom gm;
    Consts k;
    int ci, tgrad;
    int tg[4];                    // tile grid (k columns, j columns, i chunks) of a single-case launch
    // VX: Q (after the WENO sweeps), mu, the diagonal metric and J; the isothermal upper xi face
    Fields5 q;
    gcdp mu, m0, m4, m8, J;
    int iso_hi;
    double gam_iso;
};
template <int S, bool TG, bool VX = false, int GJ = ::GJ, int GK = ::GK>
__device__ __forceinline__ void march_body(const GradArgs &a, const int bx, const int by, const int bz)
{
    const CFields5 &pr = a.pr;
    const gcdp T = a.T;
    const Fields12 &gr = a.gr;
    const Geom &gm = a.gm;
    const Consts &k = a.k;
    const int ci = a.ci;
    constexpr int NF = TG ? 4 : 3;             // u, v, w (+ T for its derivatives)
    constexpr int G = (S + 1) / 2, NL = 2 * G + 1;
    constexpr int LK = GK + 2 * G, LJ = GJ + 2 * G, LP = LK * LJ;
    __shared__ double sm[NF * LP];
    const int tx = threadIdx.x % GK, ty = threadIdx.x / GK;
    const int k0 = bx * GK, j0 = by * GJ;
    const int kk = k0 + tx, jj = j0 + ty;
    const bool mine = (kk < gm.ng[2]) && (jj < gm.ng[1]);
    const int i0 = bz * ci, i1 = min(i0 + ci, gm.ng[0]);
    const gcdp src[4] = {pr.f[1], pr.f[2], pr.f[3], T};
    const long col = (long)jj * gm.st[1] + kk;
    constexpr int NT = GK * GJ, NST = (LP + NT - 1) / NT;   // staged plane elements per thread
    const int c0 = (ty + G) * LK + (tx + G);                  // this thread's node in a staged plane
    const bool jin = mine && jj >= gm.lo[1] && jj < gm.lo[1] + gm.n[1];
    const bool kin = mine && kk >= gm.lo[2] && kk < gm.lo[2] + gm.n[2];
    // Planes i0-G .. i1+G-1 pass through LDS once each (with their j/k halo): plane p gives its
    // j and k derivatives when p lies in the chunk, and its centre value enters the register
    // window of 2g+1 planes, from which the i derivative of plane p-G follows.  Planes outside
    // the padded extent are clamped; they only reach windows of ghost planes, whose i derivatives
    // are not written.
    double nxt[NST][NF];
    auto fetch = [&](const int p) {
        const long pbase = (long)max(0, min(p, gm.ng[0] - 1)) * gm.st[0];
#pragma unroll
        for (int s = 0; s < NST; s++) {
            const int e = threadIdx.x + s * NT;
            const int lj = e / LK, lk = e - lj * LK;
            const int j = j0 - G + lj, kq = k0 - G + lk;
            const bool in = (e < LP) && (j >= 0) && (j < gm.ng[1]) && (kq >= 0) && (kq < gm.ng[2]);
            const long m = pbase + (long)j * gm.st[1] + kq;
#pragma unroll
            for (int f = 0; f < NF; f++) nxt[s][f] = in ? src[f][m] : 0.0;
        }
    };
    double win[NF][NL];
#pragma unroll
    for (int l = 0; l < NL; l++)
#pragma unroll
        for (int f = 0; f < NF; f++) win[f][l] = 0.0;
    // VX rings over the last 2g planes (index 2G-1 = plane p): T and the cross derivatives
    // v_eta, u_eta, w_zeta, u_zeta (the xi sweep's cross slots 0..3); mu and metric of planes
    // i and i+1 of the face; the previous face's flux
    constexpr int NR = VX ? 2 * G : 1;
    double tw[NR], cw[4][NR];
    double mv0[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, mv1[5] = {0.0, 0.0, 0.0, 0.0, 0.0};   // mu, m0, m4, m8, J
    double fprev[4] = {0.0, 0.0, 0.0, 0.0};
    if constexpr (VX) {
#pragma unroll
        for (int l = 0; l < NR; l++) {
            tw[l] = 0.0;
#pragma unroll
            for (int c = 0; c < 4; c++) cw[c][l] = 0.0;
        }
    }
    const bool vcol = VX && jin && kin;
    const int ilo = gm.lo[0], ihi = gm.lo[0] + gm.n[0];
    // the next plane is prefetched where the registers allow it (WENO5 order, no T derivatives)
    constexpr bool PF = (S == 5) && !TG;
    const int pend = i1 + G;
    if constexpr (PF) fetch(i0 - G);
    for (int p = i0 - G; p < pend; p++) {
        if constexpr (PF) {
#pragma unroll
            for (int s = 0; s < NST; s++) {
                const int e = threadIdx.x + s * NT;
                if (e < LP) {
#pragma unroll
                    for (int f = 0; f < NF; f++) sm[f * LP + e] = nxt[s][f];
                }
            }
        } else {
            const long pbase = (long)max(0, min(p, gm.ng[0] - 1)) * gm.st[0];
            for (int e = threadIdx.x; e < LP; e += NT) {
                const int lj = e / LK, lk = e - lj * LK;
                const int j = j0 - G + lj, kq = k0 - G + lk;
                const bool in = (j >= 0) && (j < gm.ng[1]) && (kq >= 0) && (kq < gm.ng[2]);
                const long m = pbase + (long)j * gm.st[1] + kq;
#pragma unroll
                for (int f = 0; f < NF; f++) sm[f * LP + e] = in ? src[f][m] : 0.0;
            }
        }
        __syncthreads();
        if constexpr (PF) {
            if (p + 1 < pend) fetch(p + 1);
        }
#pragma unroll
        for (int l = 0; l < NL - 1; l++)
#pragma unroll
            for (int f = 0; f < NF; f++) win[f][l] = win[f][l + 1];
#pragma unroll
        for (int f = 0; f < NF; f++) win[f][NL - 1] = sm[f * LP + c0];
        if (mine) {
            const bool chunk = (p >= i0 && p < i1);
            const long n = (long)p * gm.st[0] + col;
            if (jin && (chunk || vcol)) {
                double d[NF] = {};
#pragma unroll
                for (int l = 0; l < NL; l++)
#pragma unroll
                    for (int f = 0; f < NF; f++) d[f] += k.zd_der[l] * sm[f * LP + c0 + (l - G) * LK];
                if (chunk) {
                    if (!VX) gr.f[1][n] = d[0];
                    gr.f[4][n] = d[1]; gr.f[7][n] = d[2];
                    if constexpr (TG) gr.f[10][n] = d[3];
                }
                if constexpr (VX) {
#pragma unroll
                    for (int l = 0; l < NR - 1; l++) { cw[0][l] = cw[0][l + 1]; cw[1][l] = cw[1][l + 1]; }
                    cw[0][NR - 1] = d[1];   // v_eta
                    cw[1][NR - 1] = d[0];   // u_eta
                }
            }
            if (kin && (chunk || vcol)) {
                double d[NF] = {};
#pragma unroll
                for (int l = 0; l < NL; l++)
#pragma unroll
                    for (int f = 0; f < NF; f++) d[f] += k.zd_der[l] * sm[f * LP + c0 + (l - G)];
                if (chunk) {
                    if (!VX) gr.f[2][n] = d[0];
                    gr.f[5][n] = d[1]; gr.f[8][n] = d[2];
                    if constexpr (TG) gr.f[11][n] = d[3];
                }
                if constexpr (VX) {
#pragma unroll
                    for (int l = 0; l < NR - 1; l++) { cw[2][l] = cw[2][l + 1]; cw[3][l] = cw[3][l + 1]; }
                    cw[2][NR - 1] = d[2];   // w_zeta
                    cw[3][NR - 1] = d[0];   // u_zeta
                }
            }
            const int i = p - G;
            double gx[NF] = {};         // i derivatives of node i
            const bool iout = (i >= i0 && i >= gm.lo[0] && i < gm.lo[0] + gm.n[0]);
            if (iout) {
                const long ni = (long)i * gm.st[0] + col;
#pragma unroll
                for (int l = 0; l < NL; l++)
#pragma unroll
                    for (int f = 0; f < NF; f++) gx[f] += k.zd_der[l] * win[f][l];
                gr.f[0][ni] = gx[0]; gr.f[3][ni] = gx[1]; gr.f[6][ni] = gx[2];
                if constexpr (TG) gr.f[9][ni] = gx[3];
            }
            if constexpr (VX) {
                if (vcol) {
                    // T of plane p; mu and metric of plane i+1 (the face's upper node).  Loading
                    // these and Q one plane ahead was measured slower at 256^3 (0.95 -> 1.03 ms)
                    const long pc = (long)max(0, min(p, gm.ng[0] - 1)) * gm.st[0] + col;
#pragma unroll
                    for (int l = 0; l < NR - 1; l++) tw[l] = tw[l + 1];
                    tw[NR - 1] = T[pc];
                    const long pm = (long)max(0, min(i + 1, gm.ng[0] - 1)) * gm.st[0] + col;
#pragma unroll
                    for (int c = 0; c < 5; c++) mv0[c] = mv1[c];
                    mv1[0] = a.mu[pm]; mv1[1] = a.m0[pm]; mv1[2] = a.m4[pm]; mv1[3] = a.m8[pm]; mv1[4] = a.J[pm];
                    if (i >= max(i0, ilo) - 1 && i < min(i1, ihi)) {
                        // face i+1/2 from planes i-G+1 .. i+G: window slots 1..2G, ring slots 0..2G-1
                        double own4[4] = {0.0, 0.0, 0.0, 0.0}, cr[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int l = 0; l <= S; l++) {
                            const double cm = k.zd_mid[l], cint = k.zd_int[l];
                            own4[0] += cm * win[0][l + 1];
                            own4[1] += cm * win[1][l + 1];
                            own4[2] += cm * win[2][l + 1];
                            own4[3] += cm * tw[l];
#pragma unroll
                            for (int c = 0; c < 4; c++) cr[c] += cint * cw[c][l];
                        }
                        double dd[12];
#pragma unroll
                        for (int s2 = 0; s2 < 12; s2++) dd[s2] = 0.0;
                        dd[0 * 3 + 0] = own4[0]; dd[1 * 3 + 0] = own4[1]; dd[2 * 3 + 0] = own4[2]; dd[9 + 0] = own4[3];
                        dd[1 * 3 + 1] = cr[0]; dd[0 * 3 + 1] = cr[1];
                        dd[2 * 3 + 2] = cr[2]; dd[0 * 3 + 2] = cr[3];
                        const double g0[3] = {mv0[1], mv0[2], mv0[3]}, g1[3] = {mv1[1], mv1[2], mv1[3]};
                        double F[4];
                        face_flux_diag<0>(dd, g0, mv0[4], g1, mv1[4], mv0[0], mv1[0], F);
                        if (i >= max(i0, ilo)) {
                            // node i: faces i-1/2 (fprev) and i+1/2
                            const long ni = (long)i * gm.st[0] + col;
                            double dF[4];
#pragma unroll
                            for (int m = 0; m < 4; m++) dF[m] = F[m] - fprev[m];
                            double g[9];
                            g[0] = gx[0]; g[3] = gx[1]; g[6] = gx[2];
                            // cross derivatives of node i: ring slot G-1 (plane i)
                            g[1 * 3 + 1] = cw[0][G - 1]; g[0 * 3 + 1] = cw[1][G - 1];
                            g[2 * 3 + 2] = cw[2][G - 1]; g[0 * 3 + 2] = cw[3][G - 1];
                            g[1 * 3 + 2] = 0.0; g[2 * 3 + 1] = 0.0;
                            const double gmv[3] = {mv0[1], mv0[2], mv0[3]};
                            const double prod = node_prod_diag<0>(g, gmv, mv0[4], mv0[0]);
                            const double work = win[0][G] * dF[0] + win[1][G] * dF[1] + win[2][G] * dF[2];
                            double q0[5];
#pragma unroll
                            for (int m = 1; m < 5; m++) q0[m] = a.q.f[m][ni];
                            a.q.f[1][ni] = q0[1] + k.psi * dF[0];
                            a.q.f[2][ni] = q0[2] + k.psi * dF[1];
                            a.q.f[3][ni] = q0[3] + k.psi * dF[2];
                            const double gh = (a.iso_hi && i == ihi - 1) ? a.gam_iso : k.gam_heat;
                            a.q.f[4][ni] = q0[4] + (gh * dF[3] + k.psi * (work + prod));
                        }
#pragma unroll
                        for (int m = 0; m < 4; m++) fprev[m] = F[m];
                    }
                }
            }
        }
        __syncthreads();
    }
}
template <int S, bool TG>
__global__ __launch_bounds__(GK * GJ) void k_visc_grad_march(GradArgs a)
{
    int bx, by, bz;
    sweep_tile(blockIdx.x, a.tg, bx, by, bz);
    march_body<S, TG>(a, bx, by, bz);
}
// the march with the viscous xi direction (3D diagonal metric): 64 x 8 columns, whose 512 threads
// hold the rings in registers (201 VGPRs, two waves per SIMD).  Measured against it at 256^3: 64 x
// 16 columns spill 160 VGPRs, and 64 x 4 held to three waves per SIMD spills 60 and is slower than
// the fused zeta kernel.
constexpr int GKX = 64, GJX = 8;
template <int S>
__global__ __launch_bounds__(GKX * GJX) void k_visc_grad_march_xi(GradArgs a)
{
    int bx, by, bz;
    sweep_tile(blockIdx.x, a.tg, bx, by, bz);
    march_body<S, false, true, GJX, GKX>(a, bx, by, bz);
}

// ---- 2D stage in one kernel -------------------------------------------------------------------------
// A block owns 15 x 15 nodes and does the whole stage for them: both WENO sweeps, both viscous sweeps with
// their nodal derivatives, the source and the stage update.  Threads 0-255 sweep xi, 256-511 eta, at the
// same time and through the same code (a half's argument record is uniform per wave); 15 rows of 16
// interfaces fill 240 of 256 threads.  Periodic cases read ghosts at their image and form T and mu from
// what they read, so their stages need no ghost fill.
// A plane of 64^2 to 200^2 nodes leaves most of the chip idle and its time is the chain of its launches:
// six dependent kernels of 7-12 us per stage, one of 17 us here (64^2 WENO5 58 -> 17 us, 211 x 157 WENO9
// 74 -> 26).  Large planes are bound by the FP64 pipe and its latency (one block per CU by LDS) and gain
// from the passes over memory between the kernels: 1000 x 768 283 -> 188 us.
constexpr int PT = 15;
struct PlaneArgs {
    WenoArgs w[2];                // the sweep records of xi and eta (Q in w[0].q)
    CFields10 met;
    gcdp T, mu;                   // stored T and mu (not wrap)
    int ng[2], lo[2], nt[2];      // padded extents, first interior node, tiles (i, j)
    long st;                      // stride along i
    int wrap, visc, update;       // update: apply the stage update, else store Q
    int flat;                     // the z entries of the xi and eta metric rows are zero
    int iso_hi[2];                // upper face of the direction is an isothermal wall (ViscArgs)
    double gam_iso;
    RkArgs rk;
};
template <int S>
constexpr int plane_visc_lds()
{
    constexpr int WD = PT + S + 1, RING = PT + 2;
    return 2 * 5 * PT * PT + 4 * WD * WD + 6 * PT * WD + 8 * RING * RING + 2 * 3 * PT * PT;
}
template <int S, bool MIX>
constexpr int plane_lds()
{
    return 2 * weno_lds<S, PT, PT + 1, -1, MIX>() > plane_visc_lds<S>() ? 2 * weno_lds<S, PT, PT + 1, -1, MIX>()
                                                                       : plane_visc_lds<S>();
}
// stress_along in 2D: d holds the derivatives of u, v, T along both directions (d[3k+b], T at 9+b) and of w
// along DIR only; the rows' z entries are zero (FLAT) or not
template <int DIR, bool FLAT>
__device__ __forceinline__ void plane_stress(const double d[12], const double m[10], double t[4])
{
    if constexpr (!FLAT) {
        stress_along<DIR>(d, m, t);
    } else {
        const double ax = m[3 * DIR], ay = m[3 * DIR + 1];
        const double ux = d[0] * m[0] + d[1] * m[3], uy = d[0] * m[1] + d[1] * m[4];
        const double vx = d[3] * m[0] + d[4] * m[3], vy = d[3] * m[1] + d[4] * m[4];
        const double p = (2. / 3.) * (ux + vy), s = uy + vx;
        t[0] = (2. * ux - p) * ax + s * ay;
        t[1] = (2. * vy - p) * ay + s * ax;
        t[2] = d[6 + DIR] * (ax * ax + ay * ay);
        t[3] = (d[9] * m[0] + d[10] * m[3]) * ax + (d[9] * m[1] + d[10] * m[4]) * ay;
    }
}
// metric and mu at ring position o
template <bool FLAT>
__device__ __forceinline__ double plane_metric(const double *MM, const int o, double m[10])
{
    constexpr int NR = (PT + 2) * (PT + 2);
#pragma unroll
    for (int c = 0; c < 10; c++) m[c] = 0.0;
    m[0] = MM[o]; m[1] = MM[NR + o]; m[3] = MM[2 * NR + o]; m[4] = MM[3 * NR + o]; m[9] = MM[4 * NR + o];
    if constexpr (!FLAT) { m[2] = MM[6 * NR + o]; m[5] = MM[7 * NR + o]; }
    return MM[5 * NR + o];
}
// Viscous terms of a half's direction (CalcViscidFluxesIn{Xi,Eta}DirectionDirectly, src/ZD.c:47-480).
template <int S, int DIR, bool FLAT>
__device__ __forceinline__ void plane_visc(const PlaneArgs &z, const int t, const int d0, const double *UV,
                                           const double *DER, const double *MM, double *QV)
{
    constexpr int G = (S + 1) / 2, WD = PT + 2 * G, RN = WD * WD, ND = PT * WD;
    const WenoArgs &a = z.w[DIR];
    const Consts &k = a.k;
    const int ta = min(t / (PT + 1), PT - 1), di = t % (PT + 1);
    // region position of the first stencil node and its step; derivative arrays of this direction (own) and
    // the other (cross): [u, v, T][...]
    const int rb = (DIR == 0) ? di * WD + ta + G : (ta + G) * WD + di, rs = (DIR == 0) ? WD : 1;
    const double *own = DER + DIR * 3 * ND, *crs = DER + (1 - DIR) * 3 * ND;
    const int cb = (DIR == 0) ? di * PT + ta : ta * WD + di, cs = (DIR == 0) ? PT : 1;
    double own4[4] = {0.0, 0.0, 0.0, 0.0}, cr[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int l = 0; l <= S; l++) {
        const double cm = k.zd_mid[l], ci = k.zd_int[l];
#pragma unroll
        for (int f = 0; f < 4; f++) own4[f] += cm * UV[f * RN + rb + l * rs];
#pragma unroll
        for (int f = 0; f < 3; f++) cr[f] += ci * crs[f * ND + cb + l * cs];
    }
    const int mb = (DIR == 0) ? di * (PT + 2) + ta + 1 : (ta + 1) * (PT + 2) + di, ms = (DIR == 0) ? PT + 2 : 1;
    double F[4], nxt[4], d[12], m0[10], m1[10], t0[4], t1[4];
#pragma unroll
    for (int q = 0; q < 12; q++) d[q] = 0.0;
#pragma unroll
    for (int f = 0; f < 4; f++) d[3 * f + DIR] = own4[f];
    d[1 - DIR] = cr[0]; d[3 + 1 - DIR] = cr[1]; d[9 + 1 - DIR] = cr[2];
    const double mu0 = plane_metric<FLAT>(MM, mb, m0), mu1 = plane_metric<FLAT>(MM, mb + ms, m1);
    plane_stress<DIR, FLAT>(d, m0, t0);
    plane_stress<DIR, FLAT>(d, m1, t1);
    const double w0 = 0.5 * (mu0 * m0[9]), w1 = 0.5 * (mu1 * m1[9]);
#pragma unroll
    for (int q = 0; q < 4; q++) F[q] = w0 * t0[q] + w1 * t1[q];
#pragma unroll
    for (int q = 0; q < 4; q++) nxt[q] = next_lane(F[q]);
    if (di < PT && t < PT * (PT + 1)) {
        const int p = rb + G * rs;
        double dF[4];
#pragma unroll
        for (int q = 0; q < 4; q++) dF[q] = nxt[q] - F[q];
        const int po = (DIR == 0) ? di * WD + ta + G : (ta + G) * PT + di;   // the node in the own-direction arrays
        const int pc = cb + G * cs;                                          // and in the cross-direction ones
        double g[12];
#pragma unroll
        for (int q = 0; q < 12; q++) g[q] = 0.0;
        g[DIR] = own[po]; g[3 + DIR] = own[ND + po];
        g[1 - DIR] = crs[pc]; g[3 + 1 - DIR] = crs[ND + pc];
        plane_stress<DIR, FLAT>(g, m1, t1);
        const double prod = (mu1 * m1[9]) * (g[DIR] * t1[0] + g[3 + DIR] * t1[1]);
        const double work = UV[p] * dF[0] + UV[RN + p] * dF[1] + UV[2 * RN + p] * dF[2];
        const double gh = (z.iso_hi[DIR] && d0 + di == a.nD - 1) ? z.gam_iso : k.gam_heat;
        const int node = (DIR == 0) ? di * PT + ta : ta * PT + di;
        QV[node] = dF[0];
        QV[PT * PT + node] = dF[1];
        QV[2 * PT * PT + node] = (gh * dF[3] + k.psi * (work + prod));
    }
}
template <int S, bool MIX>
__device__ __forceinline__ void plane_body(const PlaneArgs &z, const int tile, double *lds)
{
    constexpr int G = (S + 1) / 2, WD = PT + 2 * G, RN = WD * WD, ND = PT * WD, RING = PT + 2, NR = RING * RING;
    constexpr int NN = PT * PT, WL = weno_lds<S, PT, PT + 1, -1, MIX>();
    const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), t = threadIdx.x & 255;
    const int ti = tile / z.nt[1], tj = tile - ti * z.nt[1];
    const int ta = min(t / (PT + 1), PT - 1), di = t % (PT + 1);
    const Consts &k = z.w[0].k;
    const int i0 = z.lo[0] + ti * PT, j0 = z.lo[1] + tj * PT;    // padded index of the tile's first node
    // The update's U_n and Q_sum and, for WENO5, the viscous window are loaded before the WENO sweeps: one
    // block per CU has nothing else to overlap those loads with.  64^2 WENO5 18.8 -> 17.1 us a stage, 1000 x
    // 768 207 -> 188, 211 x 157 WENO9 27.0 -> 25.6 (with its
    // window as well 25.1, but 43 spilled registers in a batch).
    constexpr int PER = (RN + 511) / 512;
    double in[PER][12];
    auto region = [&](const int idx, int &li, int &lj) {
        li = idx / WD; lj = idx - li * WD;
        return li >= G - 1 && li <= G + PT && lj >= G - 1 && lj <= G + PT;    // holds metric and mu
    };
    auto load_window = [&]() {
        const WenoArgs &wx = z.w[0], &wy = z.w[1];
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int idx = threadIdx.x + r * 512;
            if (idx >= RN) continue;
            int li, lj;
            const bool ring = region(idx, li, lj);
            const int i = min(i0 - G + li, z.ng[0] - 1), j = min(j0 - G + lj, z.ng[1] - 1);
            const long n = (long)i * z.st + j;
            long ns = n;
            if (z.wrap) {
                ns += (long)(i < wx.oD ? wx.nD : (i >= wx.oD + wx.nD ? -wx.nD : 0)) * z.st;
                ns += (j < wy.oD ? wy.nD : (j >= wy.oD + wy.nD ? -wy.nD : 0));
            }
            in[r][0] = wx.pr.f[1][ns]; in[r][1] = wx.pr.f[2][ns]; in[r][2] = wx.pr.f[3][ns];
            if (z.wrap) {
                in[r][3] = wx.pr.f[0][ns]; in[r][4] = wx.pr.f[4][ns];
            } else {
                in[r][3] = z.T[n];
                if (ring) in[r][4] = z.mu[n];
            }
            if (ring) {
                in[r][5] = z.met.f[0][n]; in[r][6] = z.met.f[1][n]; in[r][7] = z.met.f[3][n]; in[r][8] = z.met.f[4][n];
                in[r][9] = z.met.f[9][n];
                if (!z.flat) { in[r][10] = z.met.f[2][n]; in[r][11] = z.met.f[5][n]; }
            }
        }
    };
    if (S == 5 && z.visc) load_window();
    const int ni = i0 + (int)threadIdx.x / PT, nj = j0 + (int)threadIdx.x % PT;
    const bool own = threadIdx.x < NN && ni < z.w[0].oD + z.w[0].nD && nj < z.w[1].oD + z.w[1].nD;
    RkPre pre;
    if (z.update && own) rk_preload(z.rk, (long)ni * z.st + nj, pre);
    double keep[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    weno_body<S, PT, PT + 1, -1, MIX, true, 256>(z.w[half], half ? ti : tj, 0, half ? tj : ti, lds + half * WL, keep);
    __syncthreads();
    double *const QW = lds, *const UV = QW + 2 * 5 * NN, *const DER = UV + 4 * RN, *const MM = DER + 6 * ND;
    double *const QV = MM + 8 * NR;
    if (di < PT && t < PT * (PT + 1)) {
        const int node = half ? ta * PT + di : di * PT + ta;
#pragma unroll
        for (int m = 0; m < 5; m++) QW[(half * 5 + m) * NN + node] = keep[m];
    }
    if (z.visc) {
        if (S != 5) load_window();
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int idx = threadIdx.x + r * 512;
            if (idx >= RN) continue;
            int li, lj;
            const bool ring = region(idx, li, lj);
            const double u = in[r][0], v = in[r][1], w = in[r][2];
            double T = in[r][3], mu = in[r][4];
            if (z.wrap) node_tmu(k, pressure(k, in[r][3], u, v, w, in[r][4]), in[r][3], T, mu);
            UV[idx] = u; UV[RN + idx] = v; UV[2 * RN + idx] = w; UV[3 * RN + idx] = T;
            if (ring) {
                double *const M = MM + (li - G + 1) * RING + lj - G + 1;
#pragma unroll
                for (int c = 0; c < 5; c++) M[c * NR] = in[r][5 + c];
                M[5 * NR] = mu;
                if (!z.flat) { M[6 * NR] = in[r][10]; M[7 * NR] = in[r][11]; }
            }
        }
        __syncthreads();
        // nodal derivatives of u, v, T: the half's direction at the nodes interior to it along that
        // direction, over the whole region across it
        for (int idx = t; idx < ND; idx += 256) {
            const int rb = half ? (idx / PT) * WD + idx % PT : idx, rs = half ? 1 : WD;
            double d[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int l = 0; l <= S + 1; l++) {
                const double c = k.zd_der[l];
                d[0] += c * UV[rb + l * rs];
                d[1] += c * UV[RN + rb + l * rs];
                d[2] += c * UV[3 * RN + rb + l * rs];
            }
#pragma unroll
            for (int f = 0; f < 3; f++) DER[(half * 3 + f) * ND + idx] = d[f];
        }
        __syncthreads();
        if (z.flat) {
            if (half == 0) plane_visc<S, 0, true>(z, t, ti * PT, UV, DER, MM, QV);
            else plane_visc<S, 1, true>(z, t, tj * PT, UV, DER, MM, QV + 3 * NN);
        } else {
            if (half == 0) plane_visc<S, 0, false>(z, t, ti * PT, UV, DER, MM, QV);
            else plane_visc<S, 1, false>(z, t, tj * PT, UV, DER, MM, QV + 3 * NN);
        }
    }
    __syncthreads();
    double cflv = 0.0;
    {
        const int node = threadIdx.x;
        if (own) {
            const long n = (long)ni * z.st + nj;
            double q[5];
#pragma unroll
            for (int m = 0; m < 5; m++) q[m] = QW[m * NN + node] + QW[(5 + m) * NN + node];
            if (z.visc) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    q[1] = q[1] + k.psi * QV[(h * 3 + 0) * NN + node];
                    q[2] = q[2] + k.psi * QV[(h * 3 + 1) * NN + node];
                    q[4] = q[4] + QV[(h * 3 + 2) * NN + node];
                }
            }
            if (z.update) {
                double m9[9];
#pragma unroll
                for (int c = 0; c < 9; c++) m9[c] = z.rk.cfl_red ? z.met.f[c][n] : 0.0;
                rk_point(z.rk, n, z.met.f[9][n], q, m9, &cflv, &pre);
            } else {
#pragma unroll
                for (int m = 0; m < 5; m++) z.w[0].q.f[m][n] = q[m];
            }
        }
    }
    if (z.update && z.rk.cfl_red) wave_max_to(z.rk.cfl_red, cflv);
}
template <int S, bool MIX>
__global__ __launch_bounds__(512) void k_plane(PlaneArgs z)
{
    __shared__ double lds[plane_lds<S, MIX>()];
    plane_body<S, MIX>(z, blockIdx.x, lds);
}

// ---- batched launches ----------------------------------------------------------------------------
// One launch runs a kernel class over many independent cases.  The launch's work list holds one
// descriptor per block of every case: (case, tile x, tile y, tile z), or (case, block, 0, 0) for
// the node-parallel kernels, precomputed on the host so that a block starts from one scalar load
// and no integer division.  Blocks walk the list (one item per block, or with a grid stride when
// the launch is sized to the device: persistent blocks).
// The per-case records and the work list are read-only for the launch and are addressed in the
// constant address space, as kernel arguments are: the compiler reads them with scalar loads and,
// since nothing can write them, keeps the values across the LDS fences of the sweeps instead of
// reloading them (a generic record pointer would be reloaded after every fence).
#define KCONST __attribute__((address_space(4)))
#define BATCH_PARAMS(T) const KCONST T *__restrict__ A, const KCONST int4 *__restrict__ work, const int total
template <class T>
__device__ __forceinline__ const T &rec(const KCONST T *A, const int i)
{
    return *(const T *)&A[i];
}

// P = false: one block per work item (the kernel then needs exactly the registers of its
// single-case twin); P = true: persistent blocks walking the list with a grid stride.
template <bool P, class F>
__device__ __forceinline__ void batch_walk(const int total, F &&f)
{
    if constexpr (!P) {
        if ((int)blockIdx.x < total) f((int)blockIdx.x);
    } else {
        for (int b = blockIdx.x; b < total; b += gridDim.x) {
            f(b);
            __syncthreads();
        }
    }
}

struct GhostArgs { Fields10 f; int nf; Geom gm; };
struct ValuesArgs { CFields5 pr; gdp T, mu, P, C; Geom gm; Consts k; };
template <bool P>
__global__ __launch_bounds__(256) void k_ghost_batch(BATCH_PARAMS(GhostArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        const GhostArgs &a = rec(A, w.x);
        ghost_body(a.f, a.nf, a.gm, (long)w.y * 256 + threadIdx.x);
    });
}
template <bool P>
__global__ __launch_bounds__(256) void k_values_batch(BATCH_PARAMS(ValuesArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        const ValuesArgs &a = rec(A, w.x);
        values_body(a.pr, a.T, a.mu, a.P, a.C, a.gm, a.k, (long)w.y * 256 + threadIdx.x);
    });
}
struct GhostValuesArgs { Fields5 pr; gdp T, mu, P, C; Geom gm; Consts k; };
template <bool P>
__global__ __launch_bounds__(256) void k_ghost_values_batch(BATCH_PARAMS(GhostValuesArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        const GhostValuesArgs &a = rec(A, w.x);
        ghost_values_body(a.pr, a.T, a.mu, a.P, a.C, a.gm, a.k, (long)w.y * 256 + threadIdx.x);
    });
}
template <bool P>
__global__ __launch_bounds__(256) void k_face_batch(BATCH_PARAMS(BcArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        face_body(rec(A, w.x), (long)w.y * 256 + threadIdx.x);
    });
}
template <bool P>
__global__ __launch_bounds__(256) void k_face_save_batch(BATCH_PARAMS(BcArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        face_save_body(rec(A, w.x), (long)w.y * 256 + threadIdx.x);
    });
}
struct CarryArgs { CFields5 from; Fields5 to; Geom gm; };
template <bool P>
__global__ __launch_bounds__(256) void k_carry_batch(BATCH_PARAMS(CarryArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        const CarryArgs &a = rec(A, w.x);
        carry_body(a.from, a.to, a.gm, (long)w.y * 256 + threadIdx.x);
    });
}
template <int S, bool P, bool TG>
__global__ __launch_bounds__(GK * GJ) void k_march_batch(BATCH_PARAMS(GradArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        march_body<S, TG>(rec(A, w.x), w.y, w.z, w.w);
    });
}

// derivative march kernel for an order, with or without T derivatives (the general metric), as a
// single-case launch or a batched one (persistent or not)
static const void *march_kernel(int S, bool tgrad, bool batch, bool persistent = false)
{
    if (!batch) {
        if (S == 5) return tgrad ? (const void *)&k_visc_grad_march<5, true> : (const void *)&k_visc_grad_march<5, false>;
        return tgrad ? (const void *)&k_visc_grad_march<9, true> : (const void *)&k_visc_grad_march<9, false>;
    }
    if (S == 5) {
        if (tgrad) return persistent ? (const void *)&k_march_batch<5, true, true> : (const void *)&k_march_batch<5, false, true>;
        return persistent ? (const void *)&k_march_batch<5, true, false> : (const void *)&k_march_batch<5, false, false>;
    }
    if (tgrad) return persistent ? (const void *)&k_march_batch<9, true, true> : (const void *)&k_march_batch<9, false, true>;
    return persistent ? (const void *)&k_march_batch<9, true, false> : (const void *)&k_march_batch<9, false, false>;
}

template <int S, int TA, int TDI, int AX, bool MIX, bool P>
__global__ __launch_bounds__(TA * TDI, (weno_min_waves<S, AX, MIX>())) void k_weno_batch(BATCH_PARAMS(WenoArgs))
{
    __shared__ double lds[weno_lds<S, TA, TDI, AX, MIX>()];
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        weno_body<S, TA, TDI, AX, MIX>(rec(A, w.x), w.y, w.z, w.w, lds);
    });
}

template <int S, int TA, int TDI, int AX, bool MIX, bool P>
__global__ __launch_bounds__(TA * TDI, (weno_min_waves<S, AX, MIX>())) void k_weno_last_batch(BATCH_PARAMS(WenoLastArgs))
{
    __shared__ double lds[weno_lds<S, TA, TDI, AX, MIX>()];
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        weno_last_body<S, TA, TDI, AX, MIX>(rec(A, w.x), w.y, w.z, w.w, lds);
    });
}

template <int S, int DIR, int TA, int TDI, bool DIAG, bool P>
__global__ __launch_bounds__(TA * TDI) void k_visc_batch(BATCH_PARAMS(ViscArgs))
{
    __shared__ double lds[visc_lds<S, DIR, TA, TDI, DIAG>()];
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        visc_body<S, DIR, TA, TDI, DIAG>(rec(A, w.x), w.y, w.z, w.w, lds);
    });
}
template <int S, int TA, int TDI, bool MIX, bool P>
__global__ __launch_bounds__(TA * TDI, (weno_min_waves<S, 2, MIX>())) void k_zeta_batch(BATCH_PARAMS(ZetaArgs))
{
    __shared__ double lds[zeta_lds<S, TA, TDI, MIX>()];
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        zeta_body<S, TA, TDI, MIX>(rec(A, w.x), w.y, w.z, w.w, lds);
    });
}

template <bool MIX, bool P>
__global__ __launch_bounds__(256, (MIX ? 1 : ETA_WAVES)) void k_eta_batch(BATCH_PARAMS(EtaArgs))
{
    __shared__ double lds[eta_lds<MIX>()];
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        eta_body<MIX>(rec(A, w.x), w.y, w.z, w.w, lds);
    });
}
template <int S, bool MIX, bool P>
__global__ __launch_bounds__(512) void k_plane_batch(BATCH_PARAMS(PlaneArgs))
{
    __shared__ double lds[plane_lds<S, MIX>()];
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        plane_body<S, MIX>(rec(A, w.x), w.y, lds);
    });
}
template <bool P>
__global__ __launch_bounds__(GKX * GJX) void k_march_xi_batch(BATCH_PARAMS(GradArgs))
{
    batch_walk<P>(total, [&](const int b) {
        const int4 w = rec(work, b);
        march_body<5, false, true, GJX, GKX>(rec(A, w.x), w.y, w.z, w.w);
    });
}

// Q += J * src (manufactured-solution source) for the stage residual returned by shx_rhs.
__global__ void k_add_source(Fields5 q, CFields5 src, const double *J, Geom gm)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    if (t >= nint) return;
    const int kk = (int)(t % gm.n[2]);
    const long r = t / gm.n[2];
    const int jj = (int)(r % gm.n[1]);
    const int ii = (int)(r / gm.n[1]);
    const long n = (long)(ii + gm.lo[0]) * gm.st[0] + (long)(jj + gm.lo[1]) * gm.st[1] + kk + gm.lo[2];
#pragma unroll
    for (int m = 0; m < 5; m++) {
        if (m == 3 && gm.dims == 2) continue;
        q.f[m][n] += J[n] * src.f[m][n];
    }
}

// ---- metric --------------------------------------------------------------------------------
// CreateMetric (src/Functions.c:6388-6509) on the extended coordinates.
__global__ void k_metric(const double *xe, const double *ye, const double *ze, Fields10 met, Geom gm,
                         int diag3d)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= gm.ntot) return;
    int idx[3];
    const long n = padded_node(gm, t, idx);
    const int i = idx[0], j = idx[1], k = idx[2];
    const int ne1 = gm.ng[1] + 2, ne2 = (gm.dims == 3) ? gm.ng[2] + 2 : 1;
    const int ke = (gm.dims == 3) ? k + 1 : 0;
    const long ce = ((long)(i + 1) * ne1 + (j + 1)) * ne2 + ke;
    const long sI = (long)ne1 * ne2, sJ = ne2;
    double x_xi, y_xi, z_xi, x_eta, y_eta, z_eta, x_zeta, y_zeta, z_zeta;
    x_xi = (-0.5 * xe[ce - sI] + 0.5 * xe[ce + sI]);
    y_xi = (-0.5 * ye[ce - sI] + 0.5 * ye[ce + sI]);
    x_eta = (-0.5 * xe[ce - sJ] + 0.5 * xe[ce + sJ]);
    y_eta = (-0.5 * ye[ce - sJ] + 0.5 * ye[ce + sJ]);
    if (gm.dims == 2) {
        z_xi = 0.0; z_eta = 0.0; x_zeta = 0.0; y_zeta = 0.0; z_zeta = 1.0;
    } else {
        z_xi = (-0.5 * ze[ce - sI] + 0.5 * ze[ce + sI]);
        z_eta = (-0.5 * ze[ce - sJ] + 0.5 * ze[ce + sJ]);
        x_zeta = (-0.5 * xe[ce - 1] + 0.5 * xe[ce + 1]);
        y_zeta = (-0.5 * ye[ce - 1] + 0.5 * ye[ce + 1]);
        z_zeta = (-0.5 * ze[ce - 1] + 0.5 * ze[ce + 1]);
        if (diag3d) { y_xi = 0.0; z_xi = 0.0; x_eta = 0.0; z_eta = 0.0; x_zeta = 0.0; y_zeta = 0.0; }
    }
    const double J = x_xi * y_eta * z_zeta + x_eta * y_zeta * z_xi + x_zeta * y_xi * z_eta
                   - x_zeta * y_eta * z_xi - x_eta * y_xi * z_zeta - x_xi * y_zeta * z_eta;
    met.f[9][n] = J;
    met.f[0][n] = (y_eta * z_zeta - y_zeta * z_eta) / J;
    met.f[1][n] = (x_zeta * z_eta - x_eta * z_zeta) / J;
    met.f[2][n] = (x_eta * y_zeta - x_zeta * y_eta) / J;
    met.f[3][n] = (y_zeta * z_xi - y_xi * z_zeta) / J;
    met.f[4][n] = (x_xi * z_zeta - x_zeta * z_xi) / J;
    met.f[5][n] = (x_zeta * y_xi - x_xi * y_zeta) / J;
    met.f[6][n] = (y_xi * z_eta - y_eta * z_xi) / J;
    met.f[7][n] = (x_eta * z_xi - x_xi * z_eta) / J;
    met.f[8][n] = (x_xi * y_eta - x_eta * y_xi) / J;
}

// ---- reductions ----------------------------------------------------------------------------

// CFL spectral-radius maximum over interior nodes; positive doubles order like their bit
// patterns, so the block maxima combine with an unsigned 64-bit atomic max.
__global__ void k_cfl_max(CFields5 pr, CFields10 met, Geom gm, Consts k, unsigned long long *out)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    double v = 0.0;
    if (t < nint) {
        const int kk = (int)(t % gm.n[2]);
        const long r = t / gm.n[2];
        const int jj = (int)(r % gm.n[1]);
        const int ii = (int)(r / gm.n[1]);
        const long n = (long)(ii + gm.lo[0]) * gm.st[0] + (long)(jj + gm.lo[1]) * gm.st[1] + kk + gm.lo[2];
        double m9[9];
#pragma unroll
        for (int c = 0; c < 9; c++) m9[c] = met.f[c][n];
        v = node_cfl_sum(k.gamma, k.upsilon, gm.dims, pr.f[0][n], pr.f[1][n], pr.f[2][n], pr.f[3][n], pr.f[4][n], m9);
    }
    v = wave_max(v);
    __shared__ double red[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) red[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = 0.0;
        for (int s = 0; s < (int)(blockDim.x >> 6); s++) m = fmax(m, red[s]);
        atomicMax(out + (blockIdx.x & (RED_SLOTS - 1)), (unsigned long long)__double_as_longlong(m));
    }
}

// the maximum of the slots to a pinned host word; the slots are left clear (one block of RED_SLOTS)
__global__ __launch_bounds__(RED_SLOTS) void k_red_report(unsigned long long *red, unsigned long long *host)
{
    __shared__ double sh[RED_SLOTS / 64];
    const double v = wave_max(__longlong_as_double((long long)red[threadIdx.x]));
    red[threadIdx.x] = 0;
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = sh[0];
        for (int w = 1; w < RED_SLOTS / 64; w++) m = fmax(m, sh[w]);
        __hip_atomic_store(host, (unsigned long long)__double_as_longlong(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// checkNAN (src/Functions.c:5419-5467): count and overwrite non-finite interior rho (and the
// stored p, where it is kept).
__global__ void k_check_nan(Fields5 pr, gdp P, Geom gm, int *count)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    int bad = 0;
    if (t < nint) {
        const int kk = (int)(t % gm.n[2]);
        const long r = t / gm.n[2];
        const int jj = (int)(r % gm.n[1]);
        const int ii = (int)(r / gm.n[1]);
        const long n = (long)(ii + gm.lo[0]) * gm.st[0] + (long)(jj + gm.lo[1]) * gm.st[1] + kk + gm.lo[2];
        const double rho = pr.f[0][n];
        if (!isfinite(rho)) {
            bad = 1;
            pr.f[0][n] = 1000000; pr.f[1][n] = 1000000; pr.f[2][n] = 1000000; pr.f[3][n] = 1000000;
            if (P) P[n] = 1000000;
        }
    }
    bad = wave_sum(bad);
    if ((threadIdx.x & 63) == 0 && bad) atomicAdd(count, bad);
}

// ---- post-processing ---------------------------------------------------------------------
// lambda2 of interior node n (CalcLambda2, src/Functions.c:5846-6070): velocity derivatives as
// differences of midpoint-interpolated values (the viscous interpolation table), the Cartesian
// gradient through the metric, the middle eigenvalue of S^2 + Omega^2 by the trigonometric
// solution of the characteristic cubic, capped at 0.  The reference's strain tensor carries half
// the derivative on its diagonal (s11 = 0.5 u_x, src/Functions.c:5952-5957); kept.
__device__ double lambda2_node(const CFields5 &pr, const CFields10 &met, const Geom &gm, const Consts &k,
                               const int S, const long n)
{
    const int half = (S + 1) / 2;
    double dv[3][3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double lo[3] = {0., 0., 0.}, hi[3] = {0., 0., 0.};
        for (int m = 0; m <= S; m++) {
            const long i0 = n + (long)(m - half) * gm.st[d], i1 = i0 + gm.st[d];
#pragma unroll
            for (int q = 0; q < 3; q++) {
                lo[q] += k.zd_int[m] * pr.f[1 + q][i0];
                hi[q] += k.zd_int[m] * pr.f[1 + q][i1];
            }
        }
#pragma unroll
        for (int q = 0; q < 3; q++) dv[q][d] = hi[q] - lo[q];
    }
    const double xx = met.f[0][n], xy = met.f[1][n], xz = met.f[2][n], ex = met.f[3][n], ey = met.f[4][n];
    const double ez = met.f[5][n], zx = met.f[6][n], zy = met.f[7][n], zz = met.f[8][n];
    const double udx = dv[0][0] * xx + dv[0][1] * ex + dv[0][2] * zx, udy = dv[0][0] * xy + dv[0][1] * ey + dv[0][2] * zy;
    const double udz = dv[0][0] * xz + dv[0][1] * ez + dv[0][2] * zz;
    const double vdx = dv[1][0] * xx + dv[1][1] * ex + dv[1][2] * zx, vdy = dv[1][0] * xy + dv[1][1] * ey + dv[1][2] * zy;
    const double vdz = dv[1][0] * xz + dv[1][1] * ez + dv[1][2] * zz;
    const double wdx = dv[2][0] * xx + dv[2][1] * ex + dv[2][2] * zx, wdy = dv[2][0] * xy + dv[2][1] * ey + dv[2][2] * zy;
    const double wdz = dv[2][0] * xz + dv[2][1] * ez + dv[2][2] * zz;
    const double om12 = 0.5 * (udy - vdx), om13 = 0.5 * (udz - wdx), om23 = 0.5 * (vdz - wdy);
    const double s11 = 0.5 * (udx), s12 = 0.5 * (udy + vdx), s13 = 0.5 * (udz + wdx);
    const double s22 = 0.5 * (vdy), s23 = 0.5 * (vdz + wdy), s33 = 0.5 * (wdz);
    const double a11 = (s11 * s11 + s12 * s12 + s13 * s13) + (-om12 * om12 - om13 * om13);
    const double a12 = (s11 * s12 + s12 * s22 + s13 * s23) + (-om13 * om23);
    const double a13 = (s11 * s13 + s12 * s23 + s13 * s33) + (om12 * om23);
    const double a22 = (s12 * s12 + s22 * s22 + s23 * s23) + (-om12 * om12 - om23 * om23);
    const double a23 = (s12 * s13 + s22 * s23 + s23 * s33) + (-om12 * om13);
    const double a33 = (s13 * s13 + s23 * s23 + s33 * s33) + (-om13 * om13 - om23 * om23);
    const double f1 = -a11 - a22 - a33;
    const double f2 = -a23 * a23 - a12 * a12 - a13 * a13 + a11 * a33 + a11 * a22 + a22 * a33;
    const double f3 = -a11 * a22 * a33 + a11 * a23 * a23 + a22 * a13 * a13 + a33 * a12 * a12 - 2. * a12 * a13 * a23;
    const double p = -f1 * f1 / 3. + f2, q = 2. * f1 * f1 * f1 / 27. - f1 * f2 / 3. + f3;
    const double rrr = sqrt(fabs(p) / 3.);
    const double pi = 3.14159265358979323846;
    const double al = acos(q / (2. * rrr * rrr * rrr));
    const double l1 = -2. * rrr * cos(al / 3.) - f1 / 3, l2 = 2. * rrr * cos(pi / 3. - al / 3.) - f1 / 3;
    const double l3 = 2. * rrr * cos(pi / 3. + al / 3.) - f1 / 3;
    double lmax = (l2 >= l1) ? l2 : l1;
    if (l3 >= lmax) lmax = l3;
    double lmin = (l2 <= l1) ? l2 : l1;
    if (l3 <= lmin) lmin = l3;
    double lam = 0.;
    if (l1 == l2 || l2 == l3) lam = l2;
    if (l1 > lmin && l1 < lmax) lam = l1;
    else if (l2 > lmin && l2 < lmax) lam = l2;
    else if (l3 > lmin && l3 < lmax) lam = l3;
    return (lam >= 0.) ? 0. : lam;
}

// CalcValuesForPost (src/Functions.c:3687-3761) on interior nodes: Mach number from the stored
// pressure (U_lastStep's, which the RK update leaves one stage behind), the density "gradient" as
// the root of the sum of squares of every (central difference x metric entry) product, and
// lambda2 (3D).  out: Mach, gradRho, Lambda2 on the padded grid.
__global__ void k_post(CFields5 pr, gcdp P, CFields10 met, Fields5 out, Geom gm, Consts k, int S)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    if (t >= nint) return;
    const int kk = (int)(t % gm.n[2]);
    const long r = t / gm.n[2];
    const int jj = (int)(r % gm.n[1]);
    const int ii = (int)(r / gm.n[1]);
    const long n = (long)(ii + gm.lo[0]) * gm.st[0] + (long)(jj + gm.lo[1]) * gm.st[1] + kk + gm.lo[2];
    const double rho = pr.f[0][n], u = pr.f[1][n], v = pr.f[2][n], w = pr.f[3][n];
    out.f[0][n] = (sqrt(u * u + v * v + w * w)) / sqrt(P[n] / rho) * k.mach;
    const double dxi = (0.5 * pr.f[0][n + gm.st[0]] - 0.5 * pr.f[0][n - gm.st[0]]) / 1.0;
    const double deta = (0.5 * pr.f[0][n + gm.st[1]] - 0.5 * pr.f[0][n - gm.st[1]]) / 1.0;
    auto sq = [](const double x) { return pow(x, 2.0); };
    if (gm.dims == 2) {
        out.f[1][n] = sqrt(sq(dxi * met.f[0][n]) + sq(deta * met.f[3][n]) + sq(dxi * met.f[1][n]) + sq(deta * met.f[4][n]));
    } else {
        const double dze = (0.5 * pr.f[0][n + gm.st[2]] - 0.5 * pr.f[0][n - gm.st[2]]) / 1.0;
        out.f[1][n] = sqrt(sq(dxi * met.f[0][n]) + sq(deta * met.f[3][n]) + sq(dze * met.f[6][n])
                           + sq(dxi * met.f[1][n]) + sq(deta * met.f[4][n]) + sq(dze * met.f[7][n])
                           + sq(dxi * met.f[2][n]) + sq(deta * met.f[5][n]) + sq(dze * met.f[8][n]));
        out.f[2][n] = lambda2_node(pr, met, gm, k, S, n);
    }
}

// WriteValuesFromUToFilm (src/Functions.c:2510-2553): rho, u, v, w, p, gradRho, Mach, Lambda2 of
// the interior nodes into sample `s` of the device-resident film (interior-compact, field-major)
__global__ void k_film(CFields5 pr, gcdp P, CFields5 post, gdp film, long nint, int s, Geom gm)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nint) return;
    const int kk = (int)(t % gm.n[2]);
    const long r = t / gm.n[2];
    const int jj = (int)(r % gm.n[1]);
    const int ii = (int)(r / gm.n[1]);
    const long n = (long)(ii + gm.lo[0]) * gm.st[0] + (long)(jj + gm.lo[1]) * gm.st[1] + kk + gm.lo[2];
    const long base = (long)s * 8 * nint + t;
    film[base + 0 * nint] = pr.f[0][n];
    film[base + 1 * nint] = pr.f[1][n];
    film[base + 2 * nint] = pr.f[2][n];
    film[base + 3 * nint] = pr.f[3][n];
    film[base + 4 * nint] = P[n];
    film[base + 5 * nint] = post.f[1][n];
    film[base + 6 * nint] = post.f[0][n];
    film[base + 7 * nint] = post.f[2][n];
}

// probe histories (src/Functions.c:5381-5417): stored p and u, v, w of each probe node into row
// `row` of the history (field-major: p, u, v, w, each [nprobes][iters])
__global__ void k_probe(CFields5 pr, gcdp P, const long *idx, int np, gdp hist, int row, int iters)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= np) return;
    const long n = idx[t];
    const long base = (long)t * iters + row, fs = (long)np * iters;
    hist[base] = P[n];
    hist[base + fs] = pr.f[1][n];
    hist[base + 2 * fs] = pr.f[2][n];
    hist[base + 3 * fs] = pr.f[3][n];
}

// ErrorManufacturedSolution (src/ManufacturedSolution.c:745-790): squared deviations of rho and of
// the stored p from the exact values, each divided by the interior node count N, and their largest
// magnitudes, over the interior nodes of the last k plane (the reference's k loop starts at
// kEndReal).  Pass 1: per-block partial sums and maxima; pass 2 (one block): the totals.
__device__ __forceinline__ void block_sum_max(double &s0, double &m0, double &s1, double &m1, double *sh)
{
    const int t = threadIdx.x;
    sh[t] = s0; sh[256 + t] = m0; sh[512 + t] = s1; sh[768 + t] = m1;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            sh[t] += sh[t + w];
            sh[256 + t] = fmax(sh[256 + t], sh[256 + t + w]);
            sh[512 + t] += sh[512 + t + w];
            sh[768 + t] = fmax(sh[768 + t], sh[768 + t + w]);
        }
        __syncthreads();
    }
    s0 = sh[0]; m0 = sh[256]; s1 = sh[512]; m1 = sh[768];
}
__global__ __launch_bounds__(256) void k_mms_error(CFields5 pr, gcdp P, gcdp ex_rho, gcdp ex_p, Geom gm,
                                                  double N, gdp part)
{
    __shared__ double sh[1024];
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nplane = (long)gm.n[0] * gm.n[1];
    double s0 = 0.0, m0 = 0.0, s1 = 0.0, m1 = 0.0;
    if (t < nplane) {
        const int jj = (int)(t % gm.n[1]), ii = (int)(t / gm.n[1]);
        const long n = (long)(ii + gm.lo[0]) * gm.st[0] + (long)(jj + gm.lo[1]) * gm.st[1] + (gm.lo[2] + gm.n[2] - 1);
        const double dr = ex_rho[n] - pr.f[0][n], dp = ex_p[n] - P[n];
        s0 = (dr * dr) / N; m0 = fabs(dr);
        s1 = (dp * dp) / N; m1 = fabs(dp);
    }
    block_sum_max(s0, m0, s1, m1, sh);
    if (threadIdx.x == 0) {
        part[4 * blockIdx.x + 0] = s0; part[4 * blockIdx.x + 1] = m0;
        part[4 * blockIdx.x + 2] = s1; part[4 * blockIdx.x + 3] = m1;
    }
}
__global__ __launch_bounds__(256) void k_mms_error_total(gcdp part, int nb, gdp out)
{
    __shared__ double sh[1024];
    double s0 = 0.0, m0 = 0.0, s1 = 0.0, m1 = 0.0;
    for (int b = threadIdx.x; b < nb; b += 256) {
        s0 += part[4 * b + 0]; m0 = fmax(m0, part[4 * b + 1]);
        s1 += part[4 * b + 2]; m1 = fmax(m1, part[4 * b + 3]);
    }
    block_sum_max(s0, m0, s1, m1, sh);
    if (threadIdx.x == 0) { out[0] = sqrt(s0); out[1] = m0; out[2] = sqrt(s1); out[3] = m1; }
}

// check_Metric (src/Functions.c:6198-6243): count the padded nodes with a negative Jacobian.
__global__ void k_check_metric(gcdp J, Geom gm, int *count)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int bad = 0;
    if (t < gm.ntot) {
        int idx[3];
        const long n = padded_node(gm, t, idx);
        bad = (J[n] < 0.0) ? 1 : 0;
    }
    bad = wave_sum(bad);
    if ((threadIdx.x & 63) == 0 && bad) atomicAdd(count, bad);
}

// Rows of several device fields (pitched) to or from dense rows in pinned host memory, doubles
// [t0, t0 + n) of the fields' dense concatenation; an upload may fill further copies of each field.
// PCIe bounds both (53-57 GB/s, as a pitched DMA reaches), and one launch serves all fields.
constexpr int XFER_FIELDS = 10;
struct XferArgs {
    gdp dev[XFER_FIELDS], more[2][XFER_FIELDS];
    double *host;
    long t0, n, w, pitch, hw;     // row length, device pitch, doubles of one dense field
    int copies;                   // of `more` filled by an upload
};
__device__ __forceinline__ long xfer_index(const XferArgs &a, const long t, int &m)
{
    m = (int)(t / a.hw);
    const long r = t - (long)m * a.hw, row = r / a.w;
    return row * a.pitch + (r - row * a.w);
}
__global__ __launch_bounds__(256) void k_pack(XferArgs a)
{
    for (long q = (long)blockIdx.x * 256 + threadIdx.x; q < a.n; q += (long)gridDim.x * 256) {
        int m;
        const long n = xfer_index(a, a.t0 + q, m);
        a.host[q] = a.dev[m][n];
    }
}
__global__ __launch_bounds__(256) void k_unpack(XferArgs a)
{
    for (long q = (long)blockIdx.x * 256 + threadIdx.x; q < a.n; q += (long)gridDim.x * 256) {
        int m;
        const long n = xfer_index(a, a.t0 + q, m);
        const double v = a.host[q];
        a.dev[m][n] = v;
        if (a.copies > 0) a.more[0][m][n] = v;
        if (a.copies > 1) a.more[1][m][n] = v;
    }
}

// Plain streaming copy of n doubles (calibration of hardware byte counters).
__global__ void k_copy(const double *__restrict__ a, double *__restrict__ b, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i];
}

// ----------------------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------------------

static char g_err[512];

static int set_err(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

#define HIPCHK(call)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return set_err(SHX_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                           __FILE__, __LINE__);                                               \
    } while (0)

enum { KT_GHOST, KT_VALUES, KT_WENO0, KT_WENO1, KT_WENO2, KT_GRAD, KT_VISC0, KT_VISC1, KT_VISC2, KT_PLANE, KT_REDUCE, KT_METRIC, KT_FACES, KT_ZETA, KT_GRADXI, KT_ETA };
static const char *g_knames[SHX_NUM_KERNELS] = {
    "ghost_periodic", "ghost_values", "weno_xi", "weno_eta", "weno_zeta",
    "visc_grad", "visc_xi", "visc_eta", "visc_zeta", "plane_stage", "reduce", "metric", "ghost_faces",
    "weno_visc_zeta", "visc_grad_xi", "weno_visc_eta"};

// face kinds whose writers store a p and c that the equation of state does not give from the
// ghost's rho,u,v,w,e (subsonic outflow; the slip wall, whose ghost velocity is not the mirror's)
static bool stores_pc(const int kind)
{
    return kind == SHX_BC_OUTFLOW_NORMAL || kind == SHX_BC_OUTFLOW_RUDY || kind == SHX_BC_WALL_SLIP;
}
static bool is_wall(const int kind)
{
    return kind == SHX_BC_WALL_SLIP || kind == SHX_BC_WALL_NOSLIP || kind == SHX_BC_WALL_ISOTHERMAL;
}
// faces whose ghost metric is the mirror's (mirrorGhostCellsMetric, src/Functions.c:6849-7014) and
// whose writers cover the interior tangential range only
static bool mirrors_metric(const int kind) { return is_wall(kind) || kind == SHX_BC_FARFIELD; }
// BC_Corrector of a face's ghost nodes: slip walls reverse the momentum component along the
// face's index direction (src/BC.c:988-1172), no-slip walls all three (src/BC.c:2657-2686)
static void wall_corrector(const int kind, const int dir, double cr[3])
{
    for (int q = 0; q < 3; q++) cr[q] = 1.0;
    if (kind == SHX_BC_WALL_SLIP) cr[dir] = -1.0;
    if (kind == SHX_BC_WALL_NOSLIP || kind == SHX_BC_WALL_ISOTHERMAL) cr[0] = cr[1] = cr[2] = -1.0;
}

constexpr int STAGE_SLOTS = 4;   // staging slots of host transfers: one per host thread, two where one thread is enough

struct shx_case {
    shx_desc d;
    Geom gm;
    Consts k;
    double rk_a[4], rk_b[4], rk_q[4], rk_f[4], rk_m[4];
    hipStream_t stream;
    double *prim[3][5];    // three state buffers; cur = U_lastStep
    int cur;
    double *q[5], *qsum[5], *met[10], *grad[12], *src[5], *T, *mu;
    double *bs[6];         // exact state for manufactured faces
    double *P, *C;         // stored p and c (pc: some face is a subsonic outflow)
    double *bk[2][5];      // shx_simulate's two backups of the state (and of P), allocated on use
    double *bkP[2];
    double *post[3];       // Mach, gradRho, Lambda2 (padded), allocated on use
    double *film;          // device-resident samples: 8 interior fields each
    int last_in;           // buffer of the last stage's input of the last step (-1: none)
    long *d_probes;        // probe histories of shx_simulate
    double *hist;
    int hist_np, hist_iters;
    std::vector<double> hist_time;
    int film_cap, film_n;
    std::vector<double> film_time;
    double *PL, *RL, *UL, *C0;   // Rudy faces: step-start ghost p, rho, u; uploaded sound speed
    int pc, rudy;
    int has_src, has_metric, has_state, has_bs;
    int faces;             // number of non-periodic faces
    int needs_bs;          // some face is SHX_BC_MANUFACTURED
    int diag;              // 3D metric is diagonal (only xi_x, eta_y, zeta_z and J non-zero)
    int flat;              // 2D: xi_z and eta_z are zero (joined blocks: diag and flat of all of them)
    int wtile[3];          // WENO tile variant per direction (set by shx_tune; -1: by zeta_tile)
    unsigned long long *d_red;
    int *d_cnt;
    int *d_nan;            // running count of the fused checkNAN (shx_run, shx_run_cfl, shx_simulate)
    int nan_seen;          // the count last read
    struct HostIo { unsigned long long red; int nan; int nan_flag; double mms[4]; } *h_io;   // pinned landing slots
    int dev;               // the device current at shx_create (the stream's)
    int ncu;               // its compute units
    int st_in, st_out, st_bx, st_by;   // buffers of the step in progress (step_begin .. step_end)
    int iface;             // faces of kind SHX_BC_INTERFACE
    shx_blocks *blocks = nullptr;      // the multi-block case that holds this block
    int timing;
    std::vector<hipEvent_t> ev_pool;
    std::vector<int> ev_kind;
    size_t ev_used;
    double kt_ms[SHX_NUM_KERNELS];
    int kt_n[SHX_NUM_KERNELS];
    // the batch that holds this case (its captured step graph uses this case's state buffers as
    // they were at shx_batch_create); stepping the case alone while it is set would leave the
    // batch advancing a stale buffer
    shx_batch *batch = nullptr;
    // pinned staging of host transfers: slots of stage_len doubles (allocated by the first transfer that
    // goes through them), each with the event of the launch that last used it
    double *stage_h[STAGE_SLOTS] = {};
    hipEvent_t stage_ev[STAGE_SLOTS] = {};
    long stage_len = 0;
    int stage_threads = 0;   // host threads of a transfer, at most
};

extern "C" const char *shx_last_error(void) { return g_err; }

extern "C" int shx_device_count(int *count)
{
    if (!count) return set_err(SHX_ERR_ARG, "null count");
    HIPCHK(hipGetDeviceCount(count));
    return SHX_OK;
}

// event bracketing for per-kernel timing
static int tbeg(shx_case *c, int kind)
{
    if (!c->timing) return SHX_OK;
    if (c->ev_used + 2 > c->ev_pool.size()) {
        for (int s = 0; s < 256; s++) {
            hipEvent_t e;
            HIPCHK(hipEventCreate(&e));
            c->ev_pool.push_back(e);
            c->ev_kind.push_back(0);
        }
    }
    c->ev_kind[c->ev_used] = kind;
    HIPCHK(hipEventRecord(c->ev_pool[c->ev_used], c->stream));
    c->ev_used++;
    return SHX_OK;
}
static int tend(shx_case *c)
{
    if (!c->timing) return SHX_OK;
    c->ev_kind[c->ev_used] = -1;
    HIPCHK(hipEventRecord(c->ev_pool[c->ev_used], c->stream));
    c->ev_used++;
    return SHX_OK;
}
static int drain_events(shx_case *c)
{
    if (c->ev_used == 0) return SHX_OK;
    HIPCHK(hipStreamSynchronize(c->stream));
    for (size_t s = 0; s + 1 < c->ev_used; s += 2) {
        float ms = 0.f;
        HIPCHK(hipEventElapsedTime(&ms, c->ev_pool[s], c->ev_pool[s + 1]));
        c->kt_ms[c->ev_kind[s]] += ms;
        c->kt_n[c->ev_kind[s]] += 1;
    }
    c->ev_used = 0;
    return SHX_OK;
}
#define LAUNCH_CHECK() HIPCHK(hipGetLastError())

static inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

extern "C" int shx_create(const shx_desc *desc, shx_case **out)
{
    if (!desc || !out) return set_err(SHX_ERR_ARG, "null argument");
    *out = nullptr;
    const shx_desc &d = *desc;
    if (d.dims != 2 && d.dims != 3) return set_err(SHX_ERR_ARG, "dims must be 2 or 3 (got %d)", d.dims);
    if (d.space_order != 5 && d.space_order != 9)
        return set_err(SHX_ERR_ARG, "space_order must be 5 or 9 (got %d)", d.space_order);
    if (d.time_order != 3 && d.time_order != 4)
        return set_err(SHX_ERR_ARG, "time_order must be 3 or 4 (got %d)", d.time_order);
    if (d.precision != SHX_FP64 && d.precision != SHX_MIXED)
        return set_err(SHX_ERR_ARG, "precision must be SHX_FP64 or SHX_MIXED (got %d)", d.precision);
    for (int f = 0; f < 2 * d.dims; f++) {
        if (d.bc[f] < SHX_BC_PERIODIC || d.bc[f] > SHX_BC_INTERFACE)
            return set_err(SHX_ERR_ARG, "face %d: unknown boundary kind %d", f, d.bc[f]);
        if ((d.bc[f] == SHX_BC_PERIODIC) != (d.bc[f ^ 1] == SHX_BC_PERIODIC))
            return set_err(SHX_ERR_ARG, "faces %d and %d: a periodic face needs a periodic partner", f & ~1, f | 1);
        if ((d.bc[f] == SHX_BC_INFLOW_SUPERSONIC || d.bc[f] == SHX_BC_OUTFLOW_RIEMANN) &&
            !(d.rho_inflow > 0.0 && d.p_inflow > 0.0))
            return set_err(SHX_ERR_ARG, "face %d: inflow/outflow faces need rho_inflow > 0 and p_inflow > 0", f);
        if ((d.bc[f] == SHX_BC_OUTFLOW_NORMAL || d.bc[f] == SHX_BC_OUTFLOW_RUDY) && !(d.p_out > 0.0 && d.alpha_nonref >= 0.0))
            return set_err(SHX_ERR_ARG, "face %d: subsonic outflow faces need p_out > 0 and alpha_nonref >= 0", f);
        if (d.bc[f] == SHX_BC_WALL_ISOTHERMAL && !(d.T_wall > 0.0))
            return set_err(SHX_ERR_ARG, "face %d: isothermal walls need T_wall > 0", f);
    }
    const int S = d.space_order, g = (S + 1) / 2;
    for (int a = 0; a < d.dims; a++)
        if (d.n[a] < S + 1) return set_err(SHX_ERR_ARG, "n[%d]=%d below the stencil width %d", a, d.n[a], S + 1);
    if (!(d.gamma > 1.0) || !(d.mach > 0.0) || !(d.reynolds > 0.0) || !(d.prandtl > 0.0) || !(d.T0 > 0.0))
        return set_err(SHX_ERR_ARG, "non-physical fluid properties");

    shx_case *c = new shx_case();
    c->last_in = -1;
    c->d = d;
    Geom &gm = c->gm;
    gm.dims = d.dims;
    gm.g = g;
    for (int a = 0; a < 3; a++) {
        const bool live = (a < d.dims);
        gm.n[a] = live ? d.n[a] : 1;
        gm.ng[a] = live ? d.n[a] + S + 1 : 1;
        gm.lo[a] = live ? g : 0;
        gm.per[a] = live ? (d.bc[2 * a] == SHX_BC_PERIODIC) : 1;
        if (live && !gm.per[a]) {
            c->faces += 2;
            if (d.bc[2 * a] == SHX_BC_MANUFACTURED || d.bc[2 * a + 1] == SHX_BC_MANUFACTURED) c->needs_bs = 1;
            for (int u = 0; u < 2; u++) {
                const int kind = d.bc[2 * a + u];
                if (stores_pc(kind)) c->pc = 1;
                if (kind == SHX_BC_OUTFLOW_RUDY) c->rudy = 1;
                if (kind == SHX_BC_INTERFACE) c->iface++;
            }
        }
    }
    // rows of the contiguous axis are padded to 16 doubles (128 B) so tiles start on cache lines
    if (d.dims == 3) {
        const long pitch = ((long)gm.ng[2] + 15) / 16 * 16;
        gm.st[2] = 1; gm.st[1] = pitch; gm.st[0] = (long)gm.ng[1] * pitch;
        gm.nalloc = (long)gm.ng[0] * gm.ng[1] * pitch;
    } else {
        const long pitch = ((long)gm.ng[1] + 15) / 16 * 16;
        gm.st[2] = 1; gm.st[1] = 1; gm.st[0] = pitch;
        gm.nalloc = (long)gm.ng[0] * pitch;
    }
    gm.ntot = (long)gm.ng[0] * gm.ng[1] * gm.ng[2];
    if (gm.nalloc > (1L << 31) - 1) { delete c; return set_err(SHX_ERR_ARG, "block too large for 32-bit tiles"); }

    Consts &k = c->k;
    memset(&k, 0, sizeof k);
    k.gamma = d.gamma;
    k.upsilon = 1.0 / (d.gamma * (d.mach * d.mach));
    k.mach = d.mach;
    k.psi = 1.0 / d.reynolds;
    k.gam_heat = 1.0 / ((d.gamma - 1.0) * pow(d.mach, 2.0) * d.reynolds * d.prandtl);
    k.suth = 100.4 / d.T0;
    k.eps = d.eps_override > 0.0 ? d.eps_override : 10. * pow(DBL_MIN, 0.5);
    k.gm1_ups = (d.gamma - 1.0) / k.upsilon;
    k.igm1 = 1.0 / (d.gamma - 1.0);
    k.mms = d.manufactured ? 1 : 0;
    if (S == 9) {
        const double in9[10] = {1. / 1260., -23. / 2520., 127. / 2520., -473. / 2520., 1627. / 2520.,
                                1627. / 2520., -473. / 2520., 127. / 2520., -23. / 2520., 1. / 1260.};
        const double mi9[10] = {-3. / 9450., 351. / 75600., -2649. / 75600., 15351. / 75600., -110649. / 75600.,
                                110649. / 75600., -15351. / 75600., 2649. / 75600., -351. / 75600., 3. / 9450.};
        const double de9[11] = {-1. / 1260., 25. / 2520., -150. / 2520., 600. / 2520., -2100. / 2520., 0.,
                                2100. / 2520., -600. / 2520., 150. / 2520., -25. / 2520., 1. / 1260.};
        memcpy(k.zd_int, in9, sizeof in9); memcpy(k.zd_mid, mi9, sizeof mi9); memcpy(k.zd_der, de9, sizeof de9);
    } else {
        const double in5[6] = {1. / 60., -8. / 60., 37. / 60., 37. / 60., -8. / 60., 1. / 60.};
        const double mi5[6] = {-1. / 90., 25. / 180., -245. / 180., 245. / 180., -25. / 180., 1. / 90.};
        const double de5[7] = {-1. / 60., 3. / 20., -3. / 4., 0., 3. / 4., -3. / 20., 1. / 60.};
        memcpy(k.zd_int, in5, sizeof in5); memcpy(k.zd_mid, mi5, sizeof mi5); memcpy(k.zd_der, de5, sizeof de5);
    }
    if (d.time_order == 4) {
        const double a[4] = {1., 1., 1., 1.}, b[4] = {0., 0., 0., 0.}, q[4] = {0.5, 0.5, 1., 1. / 6.};
        const double f[4] = {0., 0., 0., 1. / 6.}, m[4] = {1., 2., 2., 0.};
        memcpy(c->rk_a, a, sizeof a); memcpy(c->rk_b, b, sizeof b); memcpy(c->rk_q, q, sizeof q);
        memcpy(c->rk_f, f, sizeof f); memcpy(c->rk_m, m, sizeof m);
    } else {
        const double a[4] = {1., 3. / 4., 1. / 3., 0.}, b[4] = {0., 1. / 4., 2. / 3., 0.};
        const double q[4] = {1., 1. / 4., 2. / 3., 0.}, z[4] = {0., 0., 0., 0.};
        memcpy(c->rk_a, a, sizeof a); memcpy(c->rk_b, b, sizeof b); memcpy(c->rk_q, q, sizeof q);
        memcpy(c->rk_f, z, sizeof z); memcpy(c->rk_m, z, sizeof z);
    }

    hipError_t e = hipGetDevice(&c->dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&c->ncu, hipDeviceAttributeMultiprocessorCount, c->dev);
    if (e == hipSuccess) e = hipStreamCreate(&c->stream);
    if (e != hipSuccess) { delete c; return set_err(SHX_ERR_HIP, "hipStreamCreate: %s", hipGetErrorString(e)); }
    const size_t bytes = sizeof(double) * (size_t)gm.nalloc;
    std::vector<double **> all;
    for (int b = 0; b < 3; b++) for (int m = 0; m < 5; m++) all.push_back(&c->prim[b][m]);
    for (int m = 0; m < 5; m++) { all.push_back(&c->q[m]); all.push_back(&c->qsum[m]); }
    for (int m = 0; m < 10; m++) all.push_back(&c->met[m]);
    for (int m = 0; m < 12; m++) all.push_back(&c->grad[m]);
    all.push_back(&c->T);
    all.push_back(&c->mu);
    if (c->pc) { all.push_back(&c->P); all.push_back(&c->C); }
    if (c->rudy) { all.push_back(&c->PL); all.push_back(&c->RL); all.push_back(&c->UL); all.push_back(&c->C0); }
    for (double **p : all) {
        e = hipMalloc((void **)p, bytes);
        if (e == hipSuccess) e = hipMemsetAsync(*p, 0, bytes, c->stream);
        if (e != hipSuccess) {
            shx_destroy(c);
            return set_err(SHX_ERR_HIP, "device allocation of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        }
    }
    e = hipMalloc((void **)&c->d_red, sizeof(unsigned long long) * RED_SLOTS);
    if (e == hipSuccess) e = hipMalloc((void **)&c->d_cnt, sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void **)&c->d_nan, sizeof(int));
    if (e == hipSuccess) e = hipMemsetAsync(c->d_nan, 0, sizeof(int), c->stream);
    if (e == hipSuccess) e = hipHostMalloc((void **)&c->h_io, sizeof(shx_case::HostIo), hipHostMallocDefault);
    if (e == hipSuccess) { memset(c->h_io, 0, sizeof(shx_case::HostIo)); e = hipStreamSynchronize(c->stream); }
    if (e != hipSuccess) { shx_destroy(c); return set_err(SHX_ERR_HIP, "setup: %s", hipGetErrorString(e)); }
    c->cur = 0;
    // WENO tiles until shx_tune times them: by zeta_tile along the contiguous axis; 16 x 16 across it, but
    // 8 x 32 across it for the diagonal metric where the sweep is not the FP64 WENO9 one: that window
    // holds 1.19 nodes per interface node against 1.40, and its LDS lets a fourth block on a CU (256^3:
    // xi sweep 0.89 -> 0.82 ms FP64, 0.93 -> 0.81 mixed; 144 x 112 x 128 mixed WENO9: 224 -> 172 and
    // 247 -> 188 us).  FP64 WENO9 and the general metric run three blocks either way and lose on eta
    // (176 x 128 x 136 WENO9 327 -> 352 us, 119 x 96 x 104 general 79 -> 91); along xi WENO9 goes either way
    // with the size (97 x 85 x 106 96 -> 106 us, 176 x 128 x 136 309 -> 302, 384^3 5.89 -> 5.32 ms).
    const bool wide = gm.dims == 3 && (d.quirks & SHX_QUIRK_METRIC_DIAG3D) && (S == 5 || d.precision == SHX_MIXED);
    for (int dir = 0; dir < 3; dir++) c->wtile[dir] = (gm.st[dir] == 1) ? -1 : (wide ? 1 : 0);
    *out = c;
    return SHX_OK;
}

extern "C" int shx_destroy(shx_case *c)
{
    if (!c) return SHX_OK;
    if (c->batch) return set_err(SHX_ERR_STATE, "the case is in a batch: destroy the batch first");
    if (c->blocks) return set_err(SHX_ERR_STATE, "the case is a block of a multi-block case: destroy that first");
    if (c->stream) hipStreamSynchronize(c->stream);
    for (int b = 0; b < 3; b++) for (int m = 0; m < 5; m++) hipFree(c->prim[b][m]);
    for (int m = 0; m < 5; m++) { hipFree(c->q[m]); hipFree(c->qsum[m]); hipFree(c->src[m]); }
    for (int m = 0; m < 10; m++) hipFree(c->met[m]);
    for (int m = 0; m < 12; m++) hipFree(c->grad[m]);
    for (int m = 0; m < 6; m++) hipFree(c->bs[m]);
    hipFree(c->T); hipFree(c->mu); hipFree(c->d_red); hipFree(c->d_cnt); hipFree(c->d_nan);
    if (c->h_io) hipHostFree(c->h_io);
    for (int b = 0; b < STAGE_SLOTS; b++) {
        if (c->stage_ev[b]) hipEventDestroy(c->stage_ev[b]);
        if (c->stage_h[b]) hipHostFree(c->stage_h[b]);
    }
    hipFree(c->P); hipFree(c->C); hipFree(c->PL); hipFree(c->RL); hipFree(c->UL); hipFree(c->C0);
    for (int b = 0; b < 2; b++) {
        for (int m = 0; m < 5; m++) hipFree(c->bk[b][m]);
        hipFree(c->bkP[b]);
    }
    for (int m = 0; m < 3; m++) hipFree(c->post[m]);
    hipFree(c->film);
    hipFree(c->d_probes);
    hipFree(c->hist);
    for (hipEvent_t e : c->ev_pool) hipEventDestroy(e);
    if (c->stream) hipStreamDestroy(c->stream);
    delete c;
    return SHX_OK;
}

extern "C" int shx_padded_extent(const shx_case *c, int ng[3])
{
    if (!c || !ng) return set_err(SHX_ERR_ARG, "null argument");
    for (int a = 0; a < 3; a++) ng[a] = c->gm.ng[a];
    return SHX_OK;
}

// Host transfers.  Host arrays use the reference layout (dense rows); device rows are padded to the
// pitch.  k_pack and k_unpack move chunks of all fields of a call between the device and slots of pinned
// memory, and host threads copy between the slots and the caller's arrays.  A state from 5 MB on takes four
// threads, each with every fourth chunk and a slot: while one copies (~14 GB/s), the launches of the others
// are on the link (53 GB/s), and no thread waits for another.  Field by field through two slots, with a
// copy's threads started per slot, the pipeline drained between fields: state downloads of 48^3 425 -> 240 us,
// 1000 x 768 1.22 -> 0.78 ms, 97 x 85 x 106 1.60 -> 1.00, 256^3 14.9 either way (PCIe).  Slots of up to 2 MB: with
// 1 MB 200^3 took 8.0 ms against 7.3, and eight threads were slower.
// A smaller state stays on the calling thread, where starting threads costs what they give (42^3 177 us
// either way, 32^3 117 against 131), through two slots, of a field or of a third of the state: the launch of
// the next chunk is in flight while it copies one.  One of up to 256 KB goes through one slot (64^2 118 -> 21 us).
// A case pins what it needs, and pinning is most of its first upload.  Eight slots of 256 KB to 2 MB for every
// case, two a thread, moved 0-2 % more per second, and a new case's first upload took 0.50 ms at 64^2, 0.80 at
// 32^3, 1.5 at 48^3, 4.0 at 97 x 85 x 106 and 2.9 at 1000 x 768 against 0.19, 0.56, 0.90, 2.6 and 2.0.
// A pitched copy straight to or from pageable memory ran at 0.3 GB/s.
constexpr long STAGE_MIN = 1L << 15, STAGE_MAX = 1L << 18;   // doubles: 256 KB, and 2 MB per slot at most
constexpr long STAGE_MANY = 5L << 17;                        // states from here on take four threads
struct Xfer {
    shx_case *c;
    XferArgs k;
    bool up;
    double *host[XFER_FIELDS];    // the caller's arrays (read only by an upload)
    long total, chunk;
    int threads, per;             // slots of a thread
};
static hipError_t xfer_launch(const Xfer &x, const long i, const int slot)
{
    XferArgs k = x.k;
    k.t0 = i * x.chunk;
    k.n = std::min(x.chunk, x.total - k.t0);
    k.host = x.c->stage_h[slot];
    const unsigned grid = (unsigned)std::min<long>((k.n + 255) / 256, 1024);
    if (x.up) k_unpack<<<grid, 256, 0, x.c->stream>>>(k);
    else k_pack<<<grid, 256, 0, x.c->stream>>>(k);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(x.c->stage_ev[slot], x.c->stream);
    return e;
}
// chunk i between its slot and the caller's arrays
static void xfer_copy(const Xfer &x, const long i, const int slot)
{
    const double *s = x.c->stage_h[slot];
    for (long t = i * x.chunk, end = std::min(t + x.chunk, x.total); t < end;) {
        const long m = t / x.k.hw, r = t - m * x.k.hw, n = std::min(x.k.hw - r, end - t);
        if (x.up) memcpy((void *)s, x.host[m] + r, sizeof(double) * n);
        else memcpy(x.host[m] + r, s, sizeof(double) * n);
        s += n;
        t += n;
    }
}
// the chunks of thread id: id, id + threads, ..., through its slots in turn
static hipError_t xfer_chunks(const Xfer &x, const int id)
{
    const long nc = (x.total + x.chunk - 1) / x.chunk;
    hipError_t e = hipSuccess;
    int slot = id * x.per;
    auto next = [&] { return (slot + 1 < (id + 1) * x.per) ? slot + 1 : id * x.per; };
    if (x.up) {
        // a slot's previous launch (of this call or an earlier one) has read it
        for (long i = id; i < nc && e == hipSuccess; i += x.threads, slot = next()) {
            if ((e = hipEventSynchronize(x.c->stage_ev[slot])) != hipSuccess) break;
            xfer_copy(x, i, slot);
            e = xfer_launch(x, i, slot);
        }
        return e;
    }
    const long ahead = (long)x.per * x.threads;
    for (long i = id; i < nc && i < id + ahead && e == hipSuccess; i += x.threads, slot = next()) e = xfer_launch(x, i, slot);
    slot = id * x.per;
    for (long i = id; i < nc && e == hipSuccess; i += x.threads, slot = next()) {
        if ((e = hipEventSynchronize(x.c->stage_ev[slot])) != hipSuccess) break;
        xfer_copy(x, i, slot);
        if (i + ahead < nc) e = xfer_launch(x, i + ahead, slot);
    }
    return e;
}
// nf fields between the device arrays dev and the caller's dense arrays host; an upload also fills the
// `copies` further arrays of each field.  A download returns with the arrays written; an upload once they
// have been read (the launches may still be in flight on the case's stream).
static int transfer(shx_case *c, const bool up, const int nf, double *const *dev, double *const *host,
                    double *const *const *more = nullptr, const int copies = 0)
{
    const Geom &gm = c->gm;
    Xfer x;
    memset(&x, 0, sizeof x);
    x.c = c;
    x.up = up;
    x.k.w = (gm.dims == 3) ? gm.ng[2] : gm.ng[1];
    x.k.pitch = (gm.dims == 3) ? gm.st[1] : gm.st[0];
    x.k.hw = gm.ntot;
    x.k.copies = copies;
    for (int m = 0; m < nf; m++) {
        if (!host[m]) return set_err(SHX_ERR_ARG, "null field pointer");
        x.k.dev[m] = dev[m];
        x.host[m] = host[m];
        for (int q = 0; q < copies; q++) x.k.more[q][m] = more[q][m];
    }
    x.total = (long)nf * gm.ntot;
    if (!c->stage_len) {
        const long state = 5 * gm.ntot;
        c->stage_threads = (state < STAGE_MANY) ? 1 : STAGE_SLOTS;
        if (state <= STAGE_MIN) c->stage_len = state;
        else if (state < STAGE_MANY) c->stage_len = std::max(gm.ntot, std::min(STAGE_MIN, (state + 2) / 3));
        else c->stage_len = std::min(STAGE_MAX, (state + 2 * STAGE_SLOTS - 1) / (2 * STAGE_SLOTS));
    }
    x.chunk = c->stage_len;
    const long nc = (x.total + x.chunk - 1) / x.chunk;
    x.threads = (int)std::min<long>(c->stage_threads, nc);
    x.per = (c->stage_threads == 1) ? 2 : 1;
    // fields that come down into one array are written in order, on one thread
    for (int m = 1; !up && m < nf; m++)
        for (int q = 0; q < m; q++)
            if (std::less<double *>()(host[q], host[m] + gm.ntot) && std::less<double *>()(host[m], host[q] + gm.ntot)) x.threads = 1;
    // the slots that xfer_chunks goes through, one allocation each: a new case's are taken from what an
    // earlier one gave back, where one of 16 MB was pinned anew
    for (int b = 0; b < x.threads * x.per && b < nc; b++) {
        if (!c->stage_h[b])
            HIPCHK(hipHostMalloc((void **)&c->stage_h[b], sizeof(double) * (size_t)c->stage_len, hipHostMallocDefault));
        if (c->stage_ev[b]) continue;
        HIPCHK(hipEventCreateWithFlags(&c->stage_ev[b], hipEventDisableTiming));
        HIPCHK(hipEventRecord(c->stage_ev[b], c->stream));
    }
    hipError_t err[STAGE_SLOTS];
    std::thread th[STAGE_SLOTS];
    for (int t = 1; t < x.threads; t++) {
        err[t] = hipErrorUnknown;
        try {
            th[t] = std::thread([&x, &err, t] {
                err[t] = hipSetDevice(x.c->dev);           // a new thread starts on device 0
                if (err[t] == hipSuccess) err[t] = xfer_chunks(x, t);
            });
        } catch (...) {
        }
    }
    err[0] = xfer_chunks(x, 0);
    for (int t = 1; t < x.threads; t++) {
        if (th[t].joinable()) th[t].join();
        else err[t] = xfer_chunks(x, t);       // no thread available: its chunks here, on the caller's device
    }
    for (int t = 0; t < x.threads; t++) HIPCHK(err[t]);
    return SHX_OK;
}
static int copy_in(shx_case *c, double *dst, const double *src)
{
    double *h = const_cast<double *>(src);
    return transfer(c, true, 1, &dst, &h);
}
static int copy_out(shx_case *c, double *dst, double *src) { return transfer(c, false, 1, &src, &dst); }

static int ghost_fill(shx_case *c, double *const *f, int nf)
{
    Fields10 ff;
    memset(&ff, 0, sizeof ff);
    for (int m = 0; m < nf; m++) ff.f[m] = f[m];
    int rc = tbeg(c, KT_GHOST);
    if (rc) return rc;
    k_ghost_periodic<<<nblk(c->gm.ntot, 256), 256, 0, c->stream>>>(ff, nf, c->gm);
    LAUNCH_CHECK();
    return tend(c);
}

// face writers of every non-periodic face, in face order (i-, i+, j-, j+, k-, k+)
// argument record of the writer of face f (f = 2 * direction + upper) in a step of length tau;
// nodes: ghost nodes it owns
static void face_args(const shx_case *c, double *const *pr, int f, double tau, BcArgs &a, long &nodes)
{
    const Geom &gm = c->gm;
    const int kind = c->d.bc[f];
    memset(&a, 0, sizeof a);
    for (int m = 0; m < 5; m++) a.pr.f[m] = pr[m];
    if (!c->d.inviscid) { a.T = c->T; a.mu = c->mu; }
    for (int m = 0; m < 6; m++) a.bs[m] = c->bs[m];
    a.kind = kind;
    a.dir = f / 2;
    a.upper = f % 2;
    a.g = gm.g;
    a.t1 = (a.dir == 0) ? 1 : 0;
    a.t2 = (a.dir == 2) ? 1 : 2;
    if (kind == SHX_BC_MANUFACTURED || mirrors_metric(kind)) {
        // interior tangential range (src/ManufacturedSolution.c:202-338, src/BC.c:804-1172)
        a.lo1 = gm.lo[a.t1]; a.n1 = gm.n[a.t1]; a.lo2 = gm.lo[a.t2]; a.n2 = gm.n[a.t2];
    } else {
        a.lo1 = 0; a.n1 = gm.ng[a.t1]; a.lo2 = 0; a.n2 = gm.ng[a.t2];
    }
    a.first = gm.lo[a.dir];
    a.last = gm.lo[a.dir] + gm.n[a.dir] - 1;
    for (int d = 0; d < 3; d++) a.st[d] = gm.st[d];
    a.rho_in = c->d.rho_inflow; a.u_in = c->d.u_inflow; a.v_in = c->d.v_inflow;
    a.w_in = c->d.w_inflow; a.p_in = c->d.p_inflow;
    a.cinf = 1.0 / c->d.mach;
    a.mach = c->d.mach;
    a.T_wall = c->d.T_wall;
    for (int m = 0; m < 9; m++) a.met[m] = c->met[m];
    a.P = c->P; a.C = c->C;
    a.PL = c->PL; a.RL = c->RL; a.UL = c->UL; a.C0 = c->C0;
    a.p_out = c->d.p_out;
    a.alpha_tau = c->d.alpha_nonref * tau;
    a.k = c->k;
    nodes = (kind == SHX_BC_PERIODIC || kind == SHX_BC_INTERFACE) ? 0 : (long)a.n1 * a.n2 * a.g;
}
static int face_fill(shx_case *c, double *const *pr, double tau)
{
    if (!c->faces) return SHX_OK;
    int rc = tbeg(c, KT_FACES);
    if (rc) return rc;
    for (int f = 0; f < 2 * c->gm.dims; f++) {
        BcArgs a;
        long nodes;
        face_args(c, pr, f, tau, a, nodes);
        if (nodes == 0) continue;
        k_face_bc<<<nblk(nodes, 256), 256, 0, c->stream>>>(a);
        LAUNCH_CHECK();
    }
    return tend(c);
}
// start of a step on state pr: keep the ghost p, rho and u of every Rudy face
static int rudy_save(shx_case *c, double *const *pr)
{
    if (!c->rudy) return SHX_OK;
    for (int f = 0; f < 2 * c->gm.dims; f++) {
        if (c->d.bc[f] != SHX_BC_OUTFLOW_RUDY) continue;
        BcArgs a;
        long nodes;
        face_args(c, pr, f, 0.0, a, nodes);
        k_face_save<<<nblk(nodes, 256), 256, 0, c->stream>>>(a);
        LAUNCH_CHECK();
    }
    return SHX_OK;
}
static int carry_ghosts(shx_case *c, double *const *from, double *const *to)
{
    if (!c->faces) return SHX_OK;
    CFields5 a;
    Fields5 b;
    for (int m = 0; m < 5; m++) { a.f[m] = from[m]; b.f[m] = to[m]; }
    int rc = tbeg(c, KT_FACES);
    if (rc) return rc;
    k_carry_ghosts<<<nblk(c->gm.ntot, 256), 256, 0, c->stream>>>(a, b, c->gm);
    LAUNCH_CHECK();
    return tend(c);
}

extern "C" int shx_build_metric(shx_case *c, const double *xe, const double *ye, const double *ze)
{
    if (!c || !xe || !ye || (c->gm.dims == 3 && !ze)) return set_err(SHX_ERR_ARG, "null argument");
    const Geom &gm = c->gm;
    const long next = (long)(gm.ng[0] + 2) * (gm.ng[1] + 2) * (gm.dims == 3 ? gm.ng[2] + 2 : 1);
    const size_t bytes = sizeof(double) * (size_t)next;
    double *dx = nullptr, *dy = nullptr, *dz = nullptr;
    HIPCHK(hipMalloc((void **)&dx, bytes));
    HIPCHK(hipMalloc((void **)&dy, bytes));
    HIPCHK(hipMalloc((void **)&dz, bytes));
    HIPCHK(hipMemcpyAsync(dx, xe, bytes, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(dy, ye, bytes, hipMemcpyHostToDevice, c->stream));
    if (gm.dims == 3) HIPCHK(hipMemcpyAsync(dz, ze, bytes, hipMemcpyHostToDevice, c->stream));
    else HIPCHK(hipMemsetAsync(dz, 0, bytes, c->stream));
    Fields10 mf;
    for (int m = 0; m < 10; m++) mf.f[m] = c->met[m];
    int rc = tbeg(c, KT_METRIC);
    if (rc) return rc;
    k_metric<<<nblk(gm.ntot, 256), 256, 0, c->stream>>>(dx, dy, dz, mf, gm,
                                                       (c->d.quirks & SHX_QUIRK_METRIC_DIAG3D) ? 1 : 0);
    LAUNCH_CHECK();
    if ((rc = tend(c))) return rc;
    if ((rc = ghost_fill(c, c->met, 10))) return rc;
    // wall and farfield faces, in face order: the ghost metric mirrored (full tangential range)
    for (int f = 0; f < 2 * gm.dims; f++) {
        if (!mirrors_metric(c->d.bc[f])) continue;
        BcArgs a;
        long nodes;
        face_args(c, c->q, f, 0.0, a, nodes);
        a.lo1 = 0; a.n1 = gm.ng[a.t1]; a.lo2 = 0; a.n2 = gm.ng[a.t2];
        nodes = (long)a.n1 * a.n2 * a.g;
        k_mirror_metric<<<nblk(nodes, 256), 256, 0, c->stream>>>(a, mf);
        LAUNCH_CHECK();
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    hipFree(dx); hipFree(dy); hipFree(dz);
    c->has_metric = 1;
    c->diag = (gm.dims == 3 && (c->d.quirks & SHX_QUIRK_METRIC_DIAG3D)) ? 1 : 0;
    c->flat = (gm.dims == 2) ? 1 : 0;
    return SHX_OK;
}

extern "C" int shx_upload_metric(shx_case *c, const double *const met[10])
{
    if (!c || !met) return set_err(SHX_ERR_ARG, "null argument");
    int rc = transfer(c, true, 10, c->met, const_cast<double *const *>(met));
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    c->has_metric = 1;
    // the diagonal-metric kernels apply when every off-diagonal entry is exactly zero
    int diag = (c->gm.dims == 3);
    static const int offd[6] = {1, 2, 3, 5, 6, 7};
    for (int s = 0; s < 6 && diag; s++)
        for (long n = 0; n < c->gm.ntot; n++)
            if (met[offd[s]][n] != 0.0) { diag = 0; break; }
    c->diag = diag;
    int flat = (c->gm.dims == 2);
    for (int s = 2; s < 6 && flat; s += 3)
        for (long n = 0; n < c->gm.ntot; n++)
            if (met[s][n] != 0.0) { flat = 0; break; }
    c->flat = flat;
    return SHX_OK;
}

extern "C" int shx_download_metric(shx_case *c, double *const met[10])
{
    if (!c || !met) return set_err(SHX_ERR_ARG, "null argument");
    int rc = transfer(c, false, 10, c->met, met);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_upload_state(shx_case *c, const double *const prim[5])
{
    if (!c || !prim) return set_err(SHX_ERR_ARG, "null argument");
    // every stage buffer gets the full array: ghost nodes that no fill writes keep these values,
    // as they do in the reference's single U_RK array
    const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
    double *const *more[2] = {c->prim[(c->cur + 1) % 3], c->prim[(c->cur + 2) % 3]};
    int rc = transfer(c, true, 5, c->prim[c->cur], const_cast<double *const *>(prim), more, 2);
    if (rc) return rc;
    if (c->pc) {
        // stored p and c of the uploaded state on every node; for Rudy faces also the step-start
        // sound speed, which stays as uploaded (the reference never recomputes U_lastStep's c)
        CFields5 cp;
        for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
        k_calc_values<<<nblk(c->gm.ntot, 256), 256, 0, c->stream>>>(cp, nullptr, nullptr, c->P, c->C, c->gm, c->k);
        LAUNCH_CHECK();
        if (c->rudy) HIPCHK(hipMemcpyAsync(c->C0, c->C, bytes, hipMemcpyDeviceToDevice, c->stream));
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->has_state = 1;
    c->last_in = -1;
    return SHX_OK;
}

extern "C" int shx_upload_boundary_state(shx_case *c, const double *const bs[6])
{
    if (!c || !bs) return set_err(SHX_ERR_ARG, "null argument");
    const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
    for (int m = 0; m < 6; m++) {
        if (!c->bs[m]) {
            HIPCHK(hipMalloc((void **)&c->bs[m], bytes));
            HIPCHK(hipMemsetAsync(c->bs[m], 0, bytes, c->stream));
        }
        int rc = copy_in(c, c->bs[m], bs[m]);
        if (rc) return rc;
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->has_bs = 1;
    return SHX_OK;
}

static int sync_ghosts(shx_case *c);
extern "C" int shx_download_state(shx_case *c, double *const prim[5])
{
    if (!c || !prim) return set_err(SHX_ERR_ARG, "null argument");
    // the ghost values the reference's U_lastStep holds after a step
    int rc0 = sync_ghosts(c);
    if (rc0) return rc0;
    int rc = transfer(c, false, 5, c->prim[c->cur], prim);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_upload_source(shx_case *c, const double *const src[5])
{
    if (!c) return set_err(SHX_ERR_ARG, "null argument");
    if (!src) { c->has_src = 0; return SHX_OK; }
    const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
    for (int m = 0; m < 5; m++) {
        if (!c->src[m]) HIPCHK(hipMalloc((void **)&c->src[m], bytes));
        int rc = copy_in(c, c->src[m], src[m]);
        if (rc) return rc;
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->has_src = 1;
    return SHX_OK;
}

// A kernel choice for one launch class: the single-case kernel, its batched twin and the tile.
struct Pick {
    const void *single, *batch, *batchp;   // single case, batched flat, batched persistent
    int TA, TDI;
};

template <int S, int TA, int TDI, int AX, bool MIX>
static Pick weno_last_pick_t()
{
    return {(const void *)&k_weno_last<S, TA, TDI, AX, MIX>, (const void *)&k_weno_last_batch<S, TA, TDI, AX, MIX, false>,
            (const void *)&k_weno_last_batch<S, TA, TDI, AX, MIX, true>, TA, TDI};
}
template <int S, int TA, int TDI, int AX, bool MIX>
static Pick weno_pick_t()
{
    return {(const void *)&k_weno<S, TA, TDI, AX, MIX>, (const void *)&k_weno_batch<S, TA, TDI, AX, MIX, false>,
            (const void *)&k_weno_batch<S, TA, TDI, AX, MIX, true>, TA, TDI};
}
// tile variants of the WENO sweeps (TA transverse x TDI along the sweep), chosen per case and
// direction by shx_tune: sweeps along the contiguous axis 4 x 64 or 8 x 32, the others 16 x 16
// or 8 x 32.  Diagonal metrics only ever use AX = 2 on the contiguous axis and 0 or 1 otherwise.
constexpr int NWTILE = 2;
template <int S, int TA, int TDI, bool MIX, bool COAL>
static Pick weno_pick_m(int ax)
{
    if constexpr (COAL) {
        if (ax == 2) return weno_last_pick_t<S, TA, TDI, 2, MIX>();
        return weno_last_pick_t<S, TA, TDI, -1, MIX>();
    } else {
        if (ax == 0) return weno_pick_t<S, TA, TDI, 0, MIX>();
        if (ax == 1) return weno_pick_t<S, TA, TDI, 1, MIX>();
        return weno_pick_t<S, TA, TDI, -1, MIX>();
    }
}
template <int S, int TA, int TDI, bool COAL>
static Pick weno_pick_s(int ax, bool mix)
{
    return mix ? weno_pick_m<S, TA, TDI, true, COAL>(ax) : weno_pick_m<S, TA, TDI, false, COAL>(ax);
}
template <int S>
static Pick weno_pick_v(bool coalesce, int variant, int ax, bool mix)
{
    if (coalesce) return variant ? weno_pick_s<S, 8, 32, true>(ax, mix) : weno_pick_s<S, 4, 64, true>(ax, mix);
    return variant ? weno_pick_s<S, 8, 32, false>(ax, mix) : weno_pick_s<S, 16, 16, false>(ax, mix);
}
// Tile along the contiguous axis for a launch over nc cases: 0 = 4 x 64, 1 = 8 x 32.  A row of 64 threads
// covers 63 nodes and one of 32 covers 31, so the last tile of a row can be nearly empty: 8 x 32 where it
// takes fewer than 7/8 of the threads.  128 x 128 x 144 inviscid (0.83 of them) 186 -> 162 us, WENO9
// viscous 176 x 128 x 136 (0.83) 523 -> 447, mixed 144 x 112 x 128 (0.83) 315 -> 298; its shorter rows read
// more halo, 256^3 WENO5 (0.90) 1.50 -> 1.53 ms, and at equal threads 97 x 85 x 106 WENO9 133 -> 136 us.
static int zeta_tile(const shx_case *const *g, const int nc)
{
    if (g[0]->wtile[2] >= 0) return g[0]->wtile[2];
    long wide = 0, narrow = 0;
    for (int i = 0; i < nc; i++) {
        const Geom &gm = g[i]->gm;
        wide += gm.n[0] * (long)nblk(gm.n[1], 4) * nblk(gm.n[2], 63);
        narrow += gm.n[0] * (long)nblk(gm.n[1], 8) * nblk(gm.n[2], 31);
    }
    return 8 * narrow < 7 * wide ? 1 : 0;
}
static Pick weno_pick(const shx_case *c, int dir, const int v)
{
    const bool diag = (c->diag && c->gm.dims == 3);
    const bool mix = (c->d.precision == SHX_MIXED);
    const bool coalesce = (c->gm.st[dir] == 1);
    const int ax = diag ? dir : -1;
    return (c->d.space_order == 5) ? weno_pick_v<5>(coalesce, v, ax, mix) : weno_pick_v<9>(coalesce, v, ax, mix);
}

// transverse axes of a sweep: A = the contiguous non-sweep axis with extent > 1, B = the other
static void sweep_axes(const Geom &gm, int dir, int &A, int &B)
{
    if (gm.dims == 3) {
        if (dir == 2) { A = 1; B = 0; } else { A = 2; B = (dir == 0) ? 1 : 0; }
    } else {
        A = (dir == 0) ? 1 : 0; B = 2;
    }
}

// The stages of an all-periodic 2D or inviscid case read ghosts at their image instead of filling them
// first (stored p and c need the fill's pass): 128 x 128 x 144 inviscid, a fill of 25 us beside sweeps of
// 444.  The viscous sweeps of a 3D case read ghosts of nodal derivatives too, which the march forms there.
static bool state_wraps(const shx_case *c)
{
    return (c->gm.dims == 2 || c->d.inviscid) && !c->faces && !c->pc;
}
static WenoArgs weno_args(const shx_case *c, double *const *pr, int dir, int first, const bool wrap = false)
{
    const Geom &gm = c->gm;
    WenoArgs a;
    memset(&a, 0, sizeof a);
    for (int m = 0; m < 5; m++) { a.pr.f[m] = pr[m]; a.q.f[m] = c->q[m]; }
    const bool diag = (c->diag && gm.dims == 3);
    if (diag) { a.m0 = c->met[4 * dir]; a.m1 = nullptr; a.m2 = nullptr; }
    else { a.m0 = c->met[3 * dir]; a.m1 = c->met[3 * dir + 1]; a.m2 = c->met[3 * dir + 2]; }
    a.J = c->met[9];
    int A, B;
    sweep_axes(gm, dir, A, B);
    a.sD = gm.st[dir]; a.sA = gm.st[A]; a.sB = gm.st[B];
    a.nD = gm.n[dir]; a.nA = gm.n[A]; a.nB = gm.n[B];
    a.oD = gm.lo[dir]; a.oA = gm.lo[A]; a.oB = gm.lo[B];
    a.ngD = gm.ng[dir];
    a.first = first;
    a.wrap = wrap ? 1 : 0;
    a.coalesce_d = (a.sD == 1);
    a.alignA = (a.sA == 1);
    a.P = c->P; a.C = c->C;
    a.pc_lo = stores_pc(c->d.bc[2 * dir]);
    a.pc_hi = stores_pc(c->d.bc[2 * dir + 1]);
    a.w_lo = is_wall(c->d.bc[2 * dir]);
    a.w_hi = is_wall(c->d.bc[2 * dir + 1]);
    wall_corrector(c->d.bc[2 * dir], dir, a.c_lo);
    wall_corrector(c->d.bc[2 * dir + 1], dir, a.c_hi);
    a.k = c->k;
    return a;
}

// tile grid of a sweep: tiles along A cover the padded span when A is contiguous (aligned rows)
static dim3 sweep_grid(int nA, int oA, int alignA, int nB, int nD, const Pick &p)
{
    const int spanA = alignA ? oA + nA : nA;
    return dim3(nblk(spanA, p.TA), nB, nblk(nD, p.TDI - 1));
}

static int launch_pick(const void *fn, dim3 grid, int threads, void *arg, hipStream_t st)
{
    void *args[] = {arg};
    HIPCHK(hipLaunchKernel(fn, grid, dim3(threads), args, 0, st));
    return SHX_OK;
}

// one-dimensional launch of a tile grid g; tg receives its extents and the tile order
static dim3 flat_grid(const dim3 g, int tg[4], int order)
{
    tg[0] = (int)g.x; tg[1] = (int)g.y; tg[2] = (int)g.z; tg[3] = order;
    return dim3(g.x * g.y * g.z);
}
// tile order of a sweep (see sweep_tile): along the sweep, except the viscous sweep of the
// slowest axis
static int sweep_order(bool visc, int dir) { return (visc && dir == 0) ? 0 : 1; }
// the last direction's record; rk: the stage update (null: Q is stored)
static WenoLastArgs weno_last_args(const shx_case *c, double *const *pr, int first, const RkArgs *rk, const bool wrap)
{
    WenoLastArgs z;
    memset(&z, 0, sizeof z);
    z.w = weno_args(c, pr, 2, first, wrap);
    for (int m = 0; m < 10; m++) z.met.f[m] = c->met[m];
    z.update = rk ? 1 : 0;
    if (rk) z.rk = *rk;
    return z;
}
// one WENO sweep along axis dir of the state `pr`; rk: the sweep is of an inviscid stage, whose last one
// (k_weno_last) applies this update
static int weno_sweep(shx_case *c, double *const *pr, int dir, int first, const RkArgs *rk = nullptr)
{
    WenoLastArgs z;
    const bool wrap = rk && state_wraps(c);      // (a residual alone: ghosts filled)
    if (dir == 2) z = weno_last_args(c, pr, first, rk, wrap);
    else z.w = weno_args(c, pr, dir, first, wrap);
    WenoArgs &a = z.w;
    const Pick p = weno_pick(c, dir, dir == 2 ? zeta_tile(&c, 1) : c->wtile[dir]);
    int rc = tbeg(c, KT_WENO0 + dir);
    if (rc) return rc;
    const dim3 grid = flat_grid(sweep_grid(a.nA, a.oA, a.alignA, a.nB, a.nD, p), a.tg, sweep_order(false, dir));
    if ((rc = launch_pick(p.single, grid, p.TA * p.TDI, dir == 2 ? (void *)&z : (void *)&a, c->stream))) return rc;
    return tend(c);
}

static int visc_sweep(shx_case *c, double *const *pr, int dir, const RkArgs *rk);
static int zeta_sweep(shx_case *c, double *const *pr, const RkArgs *rk);
// the zeta direction runs as one fused kernel (k_zeta)
static bool fuse_zeta(const shx_case *c)
{
    return c->gm.dims == 3 && c->diag && !c->d.inviscid;
}
// the viscous xi direction rides on the derivative march (k_visc_grad_march_xi; WENO5 order, whose
// rings fit the march's registers)
static bool fuse_xi(const shx_case *c)
{
    return c->gm.dims == 3 && c->diag && !c->d.inviscid && c->d.space_order == 5;
}

// the eta direction runs as one fused kernel (k_eta) where the viscous xi terms ride on the march
// and the zeta direction is fused too
static bool fuse_eta(const shx_case *c) { return fuse_xi(c) && fuse_zeta(c); }

static double iso_factor(const shx_case *c);
// (j, k) columns of a case's march, and the i planes a block of it walks.  A block (one fits on a CU)
// passes ci + 2g planes one after the other, each bound by its latency, so ci minimises rounds of
// blocks x planes per block: fewer planes where the columns alone leave CUs idle, longer chunks (fewer
// halo planes) where they fill them.  cols: the columns of all cases in the launch.  Against 32 planes
// for every size: 48^3 96 -> 22 us, 97 x 85 x 106 WENO9 136 -> 48, 119 x 96 x 104 full metric 114 -> 49,
// 176 x 128 x 136 WENO9 167 -> 130, 256^3 940 -> 866 (44 planes).
static int march_columns(const Geom &gm, const bool xi)
{
    return (int)(nblk(gm.ng[2], xi ? GKX : GK) * nblk(gm.ng[1], xi ? GJX : GJ));
}
static int march_planes(const shx_case *c, const long cols)
{
    const int n = c->gm.ng[0];
    long best = -1;
    int planes = n;
    for (int chunks = 1; chunks <= n; chunks++) {
        const int ci = (n + chunks - 1) / chunks;
        const long blocks = cols * nblk(n, ci), rounds = (blocks + c->ncu - 1) / c->ncu;
        const long cost = rounds * (ci + 2 * c->gm.g);
        if (best < 0 || cost < best) { best = cost; planes = ci; }
    }
    return planes;
}
// argument record of the 3D derivative march on stage input pr; xi: with the viscous xi terms
static GradArgs grad_args(const shx_case *c, double *const *pr, const bool xi, const int planes)
{
    GradArgs ga;
    memset(&ga, 0, sizeof ga);
    for (int m = 0; m < 5; m++) ga.pr.f[m] = pr[m];
    for (int m = 0; m < 12; m++) ga.gr.f[m] = c->grad[m];
    ga.T = c->T; ga.gm = c->gm; ga.k = c->k; ga.ci = planes; ga.tgrad = c->diag ? 0 : 1;
    if (xi) {
        for (int m = 0; m < 5; m++) ga.q.f[m] = c->q[m];
        ga.mu = c->mu; ga.m0 = c->met[0]; ga.m4 = c->met[4]; ga.m8 = c->met[8]; ga.J = c->met[9];
        ga.iso_hi = (c->d.bc[1] == SHX_BC_WALL_ISOTHERMAL) ? 1 : 0;
        ga.gam_iso = iso_factor(c);
    }
    return ga;
}
static dim3 march_grid(const Geom &gm, const bool xi, const int planes)
{
    return dim3(nblk(gm.ng[2], xi ? GKX : GK), nblk(gm.ng[1], xi ? GJX : GJ), nblk(gm.ng[0], planes));
}
// Nodal derivatives of the viscous terms.  xi: the march also adds the viscous xi terms to Q (fuse_xi
// cases, after the WENO xi sweep).
static int grad_march(shx_case *c, double *const *pr, const bool xi)
{
    const Geom &gm = c->gm;
    int rc = tbeg(c, xi ? KT_GRADXI : KT_GRAD);
    if (rc) return rc;
    const int planes = march_planes(c, march_columns(gm, xi));
    GradArgs ga = grad_args(c, pr, xi, planes);
    const void *fn = xi ? (const void *)&k_visc_grad_march_xi<5> : march_kernel(c->d.space_order, ga.tgrad, false);
    const dim3 grid = flat_grid(march_grid(gm, xi, planes), ga.tg, 0);
    void *args[] = {&ga};
    HIPCHK(hipLaunchKernel(fn, grid, dim3(xi ? GKX * GJX : GK * GJ), args, 0, c->stream));
    LAUNCH_CHECK();
    return tend(c);
}
static int eta_sweep(shx_case *c, double *const *pr);

// ---- 2D stages: one k_plane launch (after the ghost fill and the face writers, where the case has them)
static Pick plane_pick(const shx_case *c)
{
    const bool mix = (c->d.precision == SHX_MIXED);
#define SHX_PLANE_PICK(S, M) \
    Pick{(const void *)&k_plane<S, M>, (const void *)&k_plane_batch<S, M, false>, (const void *)&k_plane_batch<S, M, true>, PT, PT}
    if (c->d.space_order == 5) return mix ? SHX_PLANE_PICK(5, true) : SHX_PLANE_PICK(5, false);
    return mix ? SHX_PLANE_PICK(9, true) : SHX_PLANE_PICK(9, false);
#undef SHX_PLANE_PICK
}
// wrap: the stage input's ghosts are not filled; rk: the stage update (null: Q is stored)
static PlaneArgs plane_args(const shx_case *c, double *const *pr, const RkArgs *rk, const bool wrap)
{
    const Geom &gm = c->gm;
    PlaneArgs z;
    memset(&z, 0, sizeof z);
    for (int d = 0; d < 2; d++) {
        z.w[d] = weno_args(c, pr, d, 1, wrap);
        z.w[d].alignA = 0;
        z.ng[d] = gm.ng[d]; z.lo[d] = gm.lo[d];
        z.nt[d] = (int)nblk(gm.n[d], PT);
        z.iso_hi[d] = (c->d.bc[2 * d + 1] == SHX_BC_WALL_ISOTHERMAL) ? 1 : 0;
    }
    for (int m = 0; m < 10; m++) z.met.f[m] = c->met[m];
    z.T = c->T; z.mu = c->mu;
    z.st = gm.st[0];
    z.wrap = wrap ? 1 : 0;
    z.visc = c->d.inviscid ? 0 : 1;
    z.update = rk ? 1 : 0;
    z.flat = c->flat;
    z.gam_iso = iso_factor(c);
    if (rk) z.rk = *rk;
    return z;
}
static int plane_stage(shx_case *c, double *const *pr, const RkArgs *rk, const bool wrap)
{
    PlaneArgs z = plane_args(c, pr, rk, wrap);
    int rc = tbeg(c, KT_PLANE);
    if (rc) return rc;
    if ((rc = launch_pick(plane_pick(c).single, dim3(z.nt[0] * z.nt[1]), 512, &z, c->stream))) return rc;
    return tend(c);
}
// residual of one stage into c->q: ghost fill, derived quantities, viscous derivatives, WENO
// sweeps of every direction, then the viscous sweeps (the reference's accumulation order,
// src/Functions.c:2161-2272).  rk: when given, the stage's last kernel (2D k_plane, inviscid k_weno_last,
// else the last viscous sweep) applies this update instead of storing Q
static int stage_fluxes(shx_case *c, double *const *pr, const RkArgs *rk, double tau)
{
    const Geom &gm = c->gm;
    int rc;
    // a caller of the residual alone finds the ghosts of its state filled, as always
    const bool wrap = rk && state_wraps(c);
    if (wrap && gm.dims == 2) return plane_stage(c, pr, rk, true);
    if (wrap) {
    } else if (c->d.inviscid && !c->pc) {
        if ((rc = ghost_fill(c, pr, 5))) return rc;
    } else {
        // periodic ghosts, then T and mu (viscous) and the stored p and c (subsonic outflow faces)
        Fields5 fp;
        for (int m = 0; m < 5; m++) fp.f[m] = pr[m];
        const bool visc = !c->d.inviscid;
        if ((rc = tbeg(c, KT_VALUES))) return rc;
        k_ghost_values<<<nblk(gm.ntot, 256), 256, 0, c->stream>>>(fp, visc ? c->T : nullptr, visc ? c->mu : nullptr,
                                                                    c->P, c->C, gm, c->k);
        LAUNCH_CHECK();
        if ((rc = tend(c))) return rc;
    }
    const bool fx = fuse_xi(c);
    if ((rc = face_fill(c, pr, tau))) return rc;
    if (gm.dims == 2) return plane_stage(c, pr, rk, false);
    if (!c->d.inviscid && !fx && (rc = grad_march(c, pr, false))) return rc;
    // Q accumulates the WENO divergences, then the viscous terms; with the fused zeta direction
    // the order is WENO xi, eta, viscous xi, eta, then WENO zeta and viscous zeta together.  With
    // the viscous xi direction in the derivative march, the march runs after the WENO xi and eta
    // sweeps, in the place of the xi viscous sweep.
    // With the eta direction fused as well, the order is WENO xi, the march with viscous xi, then
    // the fused eta and zeta kernels (each WENO and viscous together).
    const bool fz = fuse_zeta(c), fe = fuse_eta(c);
    const int nsep = fz ? gm.dims - 1 : gm.dims;
    for (int dir = 0; dir < nsep; dir++) {
        if (fe && dir == 1) continue;
        if ((rc = weno_sweep(c, pr, dir, dir == 0, c->d.inviscid ? rk : nullptr))) return rc;
    }
    if (fx && (rc = grad_march(c, pr, true))) return rc;
    if (!c->d.inviscid)
        for (int dir = fx ? 1 : 0; dir < nsep; dir++) {
            if (fe && dir == 1) rc = eta_sweep(c, pr);
            else rc = visc_sweep(c, pr, dir, dir == gm.dims - 1 ? rk : nullptr);
            if (rc) return rc;
        }
    if (fz && (rc = zeta_sweep(c, pr, rk))) return rc;
    return SHX_OK;
}

template <int S, int DIR, int TA, int TDI, bool DIAG>
static Pick visc_pick_t()
{
    return {(const void *)&k_visc_sweep<S, DIR, TA, TDI, DIAG>, (const void *)&k_visc_batch<S, DIR, TA, TDI, DIAG, false>,
            (const void *)&k_visc_batch<S, DIR, TA, TDI, DIAG, true>, TA, TDI};
}

// tiles sized so that three or four blocks share a CU: diagonal metric 16 x 16 for WENO5 and 16 x 32 for
// WENO9, whose 2G = 10 halo rows make short tiles re-read most of their window (16 x 32 runs the WENO9
// xi / eta sweeps 21 % faster than 16 x 12 at 384^3; WENO5 is fastest at 16 x 16); general metric 16 x 16;
// 4 x 64 along the contiguous axis
template <int S>
static Pick visc_pick_s(int dir, bool coalesce, bool diag)
{
    constexpr int TDN = (S == 5) ? 16 : 32;
    if (coalesce) return diag ? visc_pick_t<S, 2, 4, 64, true>() : visc_pick_t<S, 2, 4, 64, false>();
    if (diag) return (dir == 0) ? visc_pick_t<S, 0, 16, TDN, true>() : visc_pick_t<S, 1, 16, TDN, true>();
    return (dir == 0) ? visc_pick_t<S, 0, 16, 16, false>() : visc_pick_t<S, 1, 16, 16, false>();
}

static Pick visc_pick(const shx_case *c, int dir)
{
    const bool diag = c->diag && c->gm.dims == 3;
    const bool coalesce = (c->gm.st[dir] == 1);
    return (c->d.space_order == 5) ? visc_pick_s<5>(dir, coalesce, diag) : visc_pick_s<9>(dir, coalesce, diag);
}

// heat-conduction factor the isothermal writer gives its ghosts (Prandtl 0.72,
// src/BC.c:2974-2976), averaged with the interior one as src/ZD.c:193-194
static double iso_factor(const shx_case *c)
{
    const shx_desc &d = c->d;
    const double gw = 1.0 / ((d.gamma - 1.0) * pow(d.mach, 2.0) * d.reynolds * 0.72);
    return 0.5 * (gw + c->k.gam_heat);
}

static ViscArgs visc_args(const shx_case *c, double *const *pr, int dir, const RkArgs *rk)
{
    const Geom &gm = c->gm;
    ViscArgs a;
    memset(&a, 0, sizeof a);
    a.u = pr[1]; a.v = pr[2]; a.w = pr[3]; a.T = c->T; a.mu = c->mu;
    const int b1 = (dir == 0) ? 1 : 0, b2 = (dir == 2) ? 1 : 2;
    const bool diag = c->diag && gm.dims == 3;
    if (diag) {
        a.cr[0] = c->grad[b1 * 3 + b1]; a.cr[1] = c->grad[dir * 3 + b1];
        a.cr[2] = c->grad[b2 * 3 + b2]; a.cr[3] = c->grad[dir * 3 + b2];
    } else {
        for (int q = 0; q < 3; q++) { a.cr[q] = c->grad[q * 3 + b1]; a.cr[4 + q] = c->grad[q * 3 + b2]; }
        a.cr[3] = c->grad[9 + b1]; a.cr[7] = c->grad[9 + b2];
    }
    for (int m = 0; m < 10; m++) a.met.f[m] = c->met[m];
    for (int m = 0; m < 5; m++) a.q.f[m] = c->q[m];
    int A, B;
    sweep_axes(gm, dir, A, B);
    a.sD = gm.st[dir]; a.sA = gm.st[A]; a.sB = gm.st[B];
    a.nD = gm.n[dir]; a.nA = gm.n[A]; a.nB = gm.n[B];
    a.oD = gm.lo[dir]; a.oA = gm.lo[A]; a.oB = gm.lo[B];
    a.ngD = gm.ng[dir];
    a.ngA = gm.ng[A];
    a.coalesce_d = (a.sD == 1);
    a.alignA = (a.sA == 1);
    a.bug = (dir == 2 && (c->d.quirks & SHX_QUIRK_ZETA_VISC_J)) ? 1 : 0;
    a.k = c->k;
    a.iso_hi = (c->d.bc[2 * dir + 1] == SHX_BC_WALL_ISOTHERMAL) ? 1 : 0;
    a.gam_iso = iso_factor(c);
    a.fuse_rk = rk ? 1 : 0;
    if (rk) a.rk = *rk;
    return a;
}

// viscous face sweep along axis dir: Q += viscous flux divergence (after the WENO sweeps)
static int visc_sweep(shx_case *c, double *const *pr, int dir, const RkArgs *rk)
{
    ViscArgs a = visc_args(c, pr, dir, rk);
    const Pick p = visc_pick(c, dir);
    int rc = tbeg(c, KT_VISC0 + dir);
    if (rc) return rc;
    const dim3 grid = flat_grid(sweep_grid(a.nA, a.oA, a.alignA, a.nB, a.nD, p), a.tg, sweep_order(true, dir));
    if ((rc = launch_pick(p.single, grid, p.TA * p.TDI, &a, c->stream))) return rc;
    return tend(c);
}
template <int S, int TA, int TDI>
static Pick zeta_pick_t(const bool mix)
{
    if (mix) return {(const void *)&k_zeta<S, TA, TDI, true>, (const void *)&k_zeta_batch<S, TA, TDI, true, false>,
                     (const void *)&k_zeta_batch<S, TA, TDI, true, true>, TA, TDI};
    return {(const void *)&k_zeta<S, TA, TDI, false>, (const void *)&k_zeta_batch<S, TA, TDI, false, false>,
            (const void *)&k_zeta_batch<S, TA, TDI, false, true>, TA, TDI};
}
static Pick zeta_pick(const shx_case *c, const int variant)
{
    const bool mix = (c->d.precision == SHX_MIXED);
    if (c->d.space_order == 5) return variant ? zeta_pick_t<5, 8, 32>(mix) : zeta_pick_t<5, 4, 64>(mix);
    return variant ? zeta_pick_t<9, 8, 32>(mix) : zeta_pick_t<9, 4, 64>(mix);
}
static ZetaArgs zeta_args(const shx_case *c, double *const *pr, const RkArgs *rk)
{
    ZetaArgs z;
    z.w = weno_args(c, pr, 2, 0);
    z.v = visc_args(c, pr, 2, rk);
    return z;
}
static int zeta_sweep(shx_case *c, double *const *pr, const RkArgs *rk)
{
    ZetaArgs z = zeta_args(c, pr, rk);
    const Pick p = zeta_pick(c, zeta_tile(&c, 1));
    int rc = tbeg(c, KT_ZETA);
    if (rc) return rc;
    const dim3 grid = flat_grid(sweep_grid(z.w.nA, z.w.oA, z.w.alignA, z.w.nB, z.w.nD, p), z.w.tg, 1);
    if ((rc = launch_pick(p.single, grid, p.TA * p.TDI, &z, c->stream))) return rc;
    return tend(c);
}

template <bool MIX>
static Pick eta_pick_t()
{
    return {(const void *)&k_eta<MIX>, (const void *)&k_eta_batch<MIX, false>, (const void *)&k_eta_batch<MIX, true>, 8, 32};
}
static Pick eta_pick(const shx_case *c)
{
    return (c->d.precision == SHX_MIXED) ? eta_pick_t<true>() : eta_pick_t<false>();
}
static EtaArgs eta_args(const shx_case *c, double *const *pr)
{
    EtaArgs z;
    z.w = weno_args(c, pr, 1, 0);
    z.v = visc_args(c, pr, 1, nullptr);
    return z;
}
static int eta_sweep(shx_case *c, double *const *pr)
{
    EtaArgs z = eta_args(c, pr);
    const Pick p = eta_pick(c);
    int rc = tbeg(c, KT_ETA);
    if (rc) return rc;
    const dim3 grid = flat_grid(sweep_grid(z.w.nA, z.w.oA, z.w.alignA, z.w.nB, z.w.nD, p), z.w.tg, 1);
    if ((rc = launch_pick(p.single, grid, p.TA * p.TDI, &z, c->stream))) return rc;
    return tend(c);
}

static RkArgs rk_args(shx_case *c, double *const *us, double *const *out, int s, double tau)
{
    RkArgs A;
    memset(&A, 0, sizeof A);
    for (int m = 0; m < 5; m++) {
        A.un.f[m] = c->prim[c->cur][m]; A.us.f[m] = us[m]; A.out.f[m] = out[m];
        A.qsum.f[m] = c->qsum[m]; A.src.f[m] = c->src[m];
    }
    A.a = c->rk_a[s]; A.b = c->rk_b[s]; A.qf = c->rk_q[s]; A.ff = c->rk_f[s]; A.mf = c->rk_m[s];
    A.tau = tau;
    A.first_stage = (s == 0);
    A.has_src = c->has_src;
    A.three = (c->gm.dims == 3);
    A.gamma = c->k.gamma;
    A.upsilon = c->k.upsilon;
    return A;
}

static int check_ready(shx_case *c)
{
    if (!c) return set_err(SHX_ERR_ARG, "null handle");
    if (!c->has_metric) return set_err(SHX_ERR_STATE, "no metric: call shx_build_metric or shx_upload_metric");
    if (!c->has_state) return set_err(SHX_ERR_STATE, "no state: call shx_upload_state");
    if (c->needs_bs && !c->has_bs)
        return set_err(SHX_ERR_STATE, "manufactured faces need shx_upload_boundary_state");
    return SHX_OK;
}

// end-of-step checks fused into the last stage's update (step_rk flags)
enum { STEP_NAN = 1, STEP_CFL = 2 };

// One time step (CalcRungeKutta and the step-end copy).  flags: STEP_NAN adds checkNAN on the new
// state to the running count c->d_nan; STEP_CFL puts the maximum node CFL sum of the new state
// into c->d_red (clear before it).
// A step in three parts, so that the blocks of a multi-block case advance stage by stage together:
// step_begin (the Rudy faces' step-start state; buffers), step_stage (one stage), step_end (the
// step-end copy).  Stage s reads buffer st_in and writes st_out; stage s+1 reads what stage s wrote
// and writes the other scratch buffer.
static int step_begin(shx_case *c)
{
    const int un = c->cur;
    c->st_bx = (un + 1) % 3;
    c->st_by = (un + 2) % 3;
    c->st_in = un;
    c->st_out = c->st_bx;
    return rudy_save(c, c->prim[un]);
}
static int step_stage(shx_case *c, int s, double tau, int flags)
{
    int rc;
    RkArgs rk = rk_args(c, c->prim[c->st_in], c->prim[c->st_out], s, tau);
    if (s == c->d.time_order - 1) {
        if (flags & STEP_NAN) { rk.nan_cnt = c->d_nan; rk.nan_flag = &c->h_io->nan_flag; rk.nanP = c->P; }
        if (flags & STEP_CFL) rk.cfl_red = c->d_red;
    }
    if ((rc = stage_fluxes(c, c->prim[c->st_in], &rk, tau))) return rc;    // its last kernel applies the update
    if ((rc = carry_ghosts(c, c->prim[c->st_in], c->prim[c->st_out]))) return rc;
    c->st_in = c->st_out;
    c->st_out = (c->st_out == c->st_bx) ? c->st_by : c->st_bx;
    return SHX_OK;
}
static void step_end(shx_case *c)
{
    // the last stage's input holds the ghost values the reference's U_RK (and so U_lastStep) keeps
    // after the step; post-processing copies them over when it needs them
    c->last_in = (c->st_in == c->st_bx) ? c->st_by : c->st_bx;
    c->cur = c->st_in;   // U_lastStep <- U_RK (pointer swap instead of WriteValuesFromU1ToU2)
}
static int step_rk(shx_case *c, double tau, int flags)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (c->batch) return set_err(SHX_ERR_STATE, "the case is in a batch: step it with shx_batch_run");
    if (c->iface) return set_err(SHX_ERR_STATE, "the case has interface faces: step it with shx_blocks_run");
    if ((rc = step_begin(c))) return rc;
    for (int s = 0; s < c->d.time_order; s++)
        if ((rc = step_stage(c, s, tau, flags))) return rc;
    step_end(c);
    return SHX_OK;
}

extern "C" int shx_calc_runge_kutta(shx_case *c, double tau) { return step_rk(c, tau, 0); }

// Non-finite densities the fused checkNAN found since the last call (synchronizes the stream).  The
// update raises the host's flag with the count, so a finite step costs no copy.
static int nan_found(shx_case *c, int &fresh)
{
    HIPCHK(hipStreamSynchronize(c->stream));
    fresh = 0;
    if (!*(volatile int *)&c->h_io->nan_flag) return SHX_OK;
    c->h_io->nan_flag = 0;
    HIPCHK(hipMemcpyAsync(&c->h_io->nan, c->d_nan, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    fresh = c->h_io->nan - c->nan_seen;
    c->nan_seen = c->h_io->nan;
    return SHX_OK;
}

// ---- multi-block cases on one device -----------------------------------------------------------
// The blocks of a case share the GPU; before every stage one gather fills the ghost layers of every
// interface face of every block from the donor blocks' stage input (the reference's
// TransferFlowParameterWithGhosts, src/Functions.c:3580-3684, whose repeated ghost-inclusive passes
// settle edges and corners).  A ghost node is followed through the faces it lies beyond, one at a
// time in axis order, periodic and interface faces first: a periodic face wraps the index, an
// interface face maps it into the donor block (normal layer l outside the face = layer l inside the
// donor's face; tangential indices through the transform).  The value is read where no such face
// is left: an interior node, or a ghost node beyond boundary-writer faces only, whose value is the
// donor's writer output of the previous stage (carried into the stage buffer), as in the reference,
// whose transfers copy the donors' ghost-inclusive planes before its writers run.  A node that is
// read is never one that is written (written nodes lie beyond an interface face), so one launch
// serves all blocks.
enum { XK_WRITER = 0, XK_PERIODIC = 1, XK_INTERFACE = 2 };
struct XRec {
    Geom gm;
    gdp f[10];            // fields moved: the stage input rho,u,v,w,e, or the metric rows and J
    int kind[6], donor[6], dface[6], tr[6][3];
    long first;           // first work item of this block
};
struct XTab {
    XRec r[SHX_BLOCKS_MAX];
    int nb, metric;
    long total;
};
__global__ __launch_bounds__(256) void k_interface_gather(XTab t)
{
    const long w = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= t.total) return;
    int b0 = 0;
    while (b0 + 1 < t.nb && w >= t.r[b0 + 1].first) b0++;
    const XRec &R0 = t.r[b0];
    const int dims = R0.gm.dims;
    int x[3];
    const long n0 = padded_node(R0.gm, w - R0.first, x);
    bool across = false;                 // a ghost in the direction of an interface face
    for (int d = 0; d < dims; d++) {
        const int lo = R0.gm.lo[d], hi = lo + R0.gm.n[d];
        if (x[d] < lo && R0.kind[2 * d] == XK_INTERFACE) across = true;
        if (x[d] >= hi && R0.kind[2 * d + 1] == XK_INTERFACE) across = true;
    }
    if (!across) return;
    int b = b0;
    int perm[3] = {0, 1, 2};             // axis of block b that each axis of block b0 runs along
    double sgn[3] = {1.0, 1.0, 1.0};
    bool moved = false;
    for (int it = 0; it < 2 * dims; it++) {
        const XRec &R = t.r[b];
        int a = -1, up = 0;
        for (int d = 0; d < dims && a < 0; d++) {
            int u = -1;
            if (x[d] < R.gm.lo[d]) u = 0;
            else if (x[d] >= R.gm.lo[d] + R.gm.n[d]) u = 1;
            if (u >= 0 && R.kind[2 * d + u] != XK_WRITER) { a = d; up = u; }
        }
        if (a < 0) break;
        moved = true;
        const int f = 2 * a + up;
        if (R.kind[f] == XK_PERIODIC) { x[a] += up ? -R.gm.n[a] : R.gm.n[a]; continue; }
        const XRec &D = t.r[R.donor[f]];
        const int fd = R.dface[f], ad = fd >> 1, dup = fd & 1;
        const int l = up ? x[a] - (R.gm.lo[a] + R.gm.n[a]) : R.gm.lo[a] - 1 - x[a];
        int y[3] = {0, 0, 0}, m[3] = {0, 1, 2};
        double s[3] = {1.0, 1.0, 1.0};
        y[ad] = dup ? D.gm.lo[ad] + D.gm.n[ad] - 1 - l : D.gm.lo[ad] + l;
        m[a] = ad;
        s[a] = (up != dup) ? 1.0 : -1.0;
        for (int q = 0; q < dims; q++) {
            if (q == a) continue;
            const int tq = R.tr[f][q], aq = (tq > 0 ? tq : -tq) - 1, r = x[q] - R.gm.lo[q];
            y[aq] = (tq > 0) ? D.gm.lo[aq] + r : D.gm.lo[aq] + D.gm.n[aq] - 1 - r;
            m[q] = aq;
            s[q] = (tq > 0) ? 1.0 : -1.0;
        }
        for (int q = 0; q < dims; q++) { sgn[q] *= s[perm[q]]; perm[q] = m[perm[q]]; }
        for (int q = 0; q < 3; q++) x[q] = y[q];
        b = R.donor[f];
    }
    if (!moved) return;
    const XRec &S = t.r[b];
    for (int d = 0; d < dims; d++)
        if (x[d] < 0 || x[d] >= S.gm.ng[d]) return;
    const long ns = (long)x[0] * S.gm.st[0] + (long)x[1] * S.gm.st[1] + (long)x[2] * S.gm.st[2];
    if (!t.metric) {
#pragma unroll
        for (int m = 0; m < 5; m++) R0.f[m][n0] = S.f[m][ns];
    } else {
        // row a of the block's metric is the donor's row perm[a], signed (src/Functions.c:2664-2686)
        for (int a = 0; a < 3; a++) {
            const int pa = (a < dims) ? perm[a] : a;
            const double sa = (a < dims) ? sgn[a] : 1.0;
#pragma unroll
            for (int c = 0; c < 3; c++) R0.f[3 * a + c][n0] = sa * S.f[3 * pa + c][ns];
        }
        R0.f[9][n0] = S.f[9][ns];
    }
}

struct shx_blocks {
    std::vector<shx_case *> b;
    int kind[SHX_BLOCKS_MAX][6], donor[SHX_BLOCKS_MAX][6], dface[SHX_BLOCKS_MAX][6], tr[SHX_BLOCKS_MAX][6][3];
    hipStream_t stream = nullptr;
    hipEvent_t ev_x = nullptr;
    std::vector<hipEvent_t> ev_b;
};

// the gather's table: the stage input buffers of every block (metric: its metric arrays)
static XTab xtab(const shx_blocks *g, bool metric)
{
    XTab t;
    memset(&t, 0, sizeof t);
    t.nb = (int)g->b.size();
    t.metric = metric ? 1 : 0;
    long first = 0;
    for (int i = 0; i < t.nb; i++) {
        const shx_case *c = g->b[i];
        XRec &r = t.r[i];
        r.gm = c->gm;
        for (int m = 0; m < 10; m++) r.f[m] = metric ? c->met[m] : (m < 5 ? c->prim[c->st_in][m] : nullptr);
        for (int f = 0; f < 6; f++) {
            r.kind[f] = g->kind[i][f]; r.donor[f] = g->donor[i][f]; r.dface[f] = g->dface[i][f];
            for (int q = 0; q < 3; q++) r.tr[f][q] = g->tr[i][f][q];
        }
        r.first = first;
        first += c->gm.ntot;
    }
    t.total = first;
    return t;
}
static int gather(shx_blocks *g, bool metric)
{
    XTab t = xtab(g, metric);
    k_interface_gather<<<nblk(t.total, 256), 256, 0, g->stream>>>(t);
    LAUNCH_CHECK();
    return SHX_OK;
}

extern "C" int shx_blocks_create(shx_case *const *blocks, int nblocks, const shx_interface *ifc, int nifc,
                                 shx_blocks **out)
{
    if (!blocks || !out || nblocks <= 0 || (nifc > 0 && !ifc) || nifc < 0) return set_err(SHX_ERR_ARG, "null argument or no blocks");
    *out = nullptr;
    if (nblocks > SHX_BLOCKS_MAX) return set_err(SHX_ERR_UNSUPPORTED, "at most %d blocks", SHX_BLOCKS_MAX);
    const shx_case *c0 = blocks[0];
    for (int i = 0; i < nblocks; i++) {
        const shx_case *c = blocks[i];
        if (!c) return set_err(SHX_ERR_ARG, "block %d is null", i);
        for (int j = 0; j < i; j++)
            if (blocks[j] == c) return set_err(SHX_ERR_ARG, "block %d appears twice", i);
        if (c->blocks || c->batch) return set_err(SHX_ERR_STATE, "block %d belongs to another group or a batch", i);
        if (c->gm.dims != c0->gm.dims || c->d.space_order != c0->d.space_order || c->d.time_order != c0->d.time_order ||
            c->d.inviscid != c0->d.inviscid)
            return set_err(SHX_ERR_ARG, "block %d: dims, scheme, RK order and viscosity must match block 0", i);
        if (c->dev != c0->dev) return set_err(SHX_ERR_ARG, "block %d is on another device", i);
    }
    const int dims = c0->gm.dims;
    shx_blocks *g = new shx_blocks();
    g->b.assign(blocks, blocks + nblocks);
    for (int i = 0; i < nblocks; i++)
        for (int f = 0; f < 6; f++) {
            const int kind = (f < 2 * dims) ? blocks[i]->d.bc[f] : SHX_BC_PERIODIC;
            g->kind[i][f] = (kind == SHX_BC_PERIODIC) ? XK_PERIODIC : (kind == SHX_BC_INTERFACE ? XK_INTERFACE : XK_WRITER);
            g->donor[i][f] = -1; g->dface[i][f] = -1;
            for (int q = 0; q < 3; q++) g->tr[i][f][q] = q + 1;
        }
    auto fail = [&](int code, const char *msg, int k) {
        delete g;
        return set_err(code, "connection %d: %s", k, msg);
    };
    for (int k = 0; k < nifc; k++) {
        const shx_interface &e = ifc[k];
        if (e.block < 0 || e.block >= nblocks || e.donor < 0 || e.donor >= nblocks) return fail(SHX_ERR_ARG, "block index out of range", k);
        if (e.face < 0 || e.face >= 2 * dims || e.donor_face < 0 || e.donor_face >= 2 * dims) return fail(SHX_ERR_ARG, "face out of range", k);
        if (g->kind[e.block][e.face] != XK_INTERFACE || g->kind[e.donor][e.donor_face] != XK_INTERFACE)
            return fail(SHX_ERR_ARG, "both faces must be of kind SHX_BC_INTERFACE", k);
        if (g->donor[e.block][e.face] >= 0) return fail(SHX_ERR_ARG, "the face is listed twice", k);
        // a signed permutation whose normal entry is the donor face's axis; whole faces
        int seen = 0;
        for (int q = 0; q < dims; q++) {
            const int t = e.transform[q], at = (t > 0 ? t : -t) - 1;
            if (at < 0 || at >= dims || (seen & (1 << at))) return fail(SHX_ERR_ARG, "transform is not a signed permutation", k);
            seen |= 1 << at;
        }
        const int a = e.face / 2, ad = e.donor_face / 2;
        if ((e.transform[a] > 0 ? e.transform[a] : -e.transform[a]) - 1 != ad)
            return fail(SHX_ERR_ARG, "the transform must take the face's normal to the donor face's", k);
        const shx_case *B = blocks[e.block], *D = blocks[e.donor];
        for (int q = 0; q < dims; q++) {
            if (q == a) continue;
            const int aq = (e.transform[q] > 0 ? e.transform[q] : -e.transform[q]) - 1;
            if (B->gm.n[q] != D->gm.n[aq]) return fail(SHX_ERR_UNSUPPORTED, "faces join only whole (tangential extents differ)", k);
        }
        if (B->gm.n[a] < B->gm.g || D->gm.n[ad] < B->gm.g) return fail(SHX_ERR_ARG, "block thinner than its ghost layers", k);
        g->donor[e.block][e.face] = e.donor;
        g->dface[e.block][e.face] = e.donor_face;
        for (int q = 0; q < 3; q++) g->tr[e.block][e.face][q] = (q < dims) ? e.transform[q] : q + 1;
    }
    for (int i = 0; i < nblocks; i++)
        for (int f = 0; f < 2 * dims; f++) {
            if (g->kind[i][f] != XK_INTERFACE) continue;
            const int d = g->donor[i][f], fd = g->dface[i][f];
            if (d < 0) { delete g; return set_err(SHX_ERR_ARG, "block %d face %d: interface without a connection", i, f); }
            if (g->donor[d][fd] != i || g->dface[d][fd] != f) {
                delete g;
                return set_err(SHX_ERR_ARG, "block %d face %d: the donor face does not connect back", i, f);
            }
            // the two sides' transforms are inverse permutations of each other
            for (int q = 0; q < dims; q++) {
                const int t = g->tr[i][f][q], aq = (t > 0 ? t : -t) - 1;
                const int back = g->tr[d][fd][aq], bq = (back > 0 ? back : -back) - 1;
                if (bq != q || (q != f / 2 && (t > 0) != (back > 0))) {
                    delete g;
                    return set_err(SHX_ERR_ARG, "block %d face %d: transforms of the two sides do not invert", i, f);
                }
            }
        }
    hipError_t e = hipStreamCreate(&g->stream);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&g->ev_x, hipEventDisableTiming);
    g->ev_b.assign(nblocks, nullptr);
    for (int i = 0; i < nblocks && e == hipSuccess; i++) e = hipEventCreateWithFlags(&g->ev_b[i], hipEventDisableTiming);
    if (e != hipSuccess) {
        shx_blocks_destroy(g);
        return set_err(SHX_ERR_HIP, "group setup: %s", hipGetErrorString(e));
    }
    for (int i = 0; i < nblocks; i++) blocks[i]->blocks = g;
    *out = g;
    return SHX_OK;
}

extern "C" int shx_blocks_destroy(shx_blocks *g)
{
    if (!g) return SHX_OK;
    if (g->stream) hipStreamSynchronize(g->stream);
    for (shx_case *c : g->b) {
        if (c->blocks == g) c->blocks = nullptr;
    }
    for (hipEvent_t ev : g->ev_b)
        if (ev) hipEventDestroy(ev);
    if (g->ev_x) hipEventDestroy(g->ev_x);
    if (g->stream) hipStreamDestroy(g->stream);
    delete g;
    return SHX_OK;
}

// the group's stream after every block's stream, and every block's after the group's
static int join_blocks(shx_blocks *g)
{
    for (size_t i = 0; i < g->b.size(); i++) {
        HIPCHK(hipEventRecord(g->ev_b[i], g->b[i]->stream));
        HIPCHK(hipStreamWaitEvent(g->stream, g->ev_b[i], 0));
    }
    return SHX_OK;
}
static int fork_blocks(shx_blocks *g)
{
    HIPCHK(hipEventRecord(g->ev_x, g->stream));
    for (shx_case *c : g->b) HIPCHK(hipStreamWaitEvent(c->stream, g->ev_x, 0));
    return SHX_OK;
}

extern "C" int shx_blocks_transfer_metric(shx_blocks *g)
{
    if (!g) return set_err(SHX_ERR_ARG, "null group");
    for (shx_case *c : g->b)
        if (!c->has_metric) return set_err(SHX_ERR_STATE, "a block has no metric yet");
    int rc;
    if ((rc = join_blocks(g)) || (rc = gather(g, true)) || (rc = fork_blocks(g))) return rc;
    HIPCHK(hipStreamSynchronize(g->stream));
    // a block's ghost rows are its neighbours' now: entries count as zero only where every block's are
    int diag = 1, flat = 1;
    for (const shx_case *c : g->b) { diag &= c->diag; flat &= c->flat; }
    for (shx_case *c : g->b) { c->diag = diag; c->flat = flat; }
    return SHX_OK;
}

extern "C" int shx_blocks_run(shx_blocks *g, double tau, int nsteps)
{
    if (!g) return set_err(SHX_ERR_ARG, "null group");
    if (nsteps < 0) return set_err(SHX_ERR_ARG, "negative step count");
    int rc;
    for (shx_case *c : g->b)
        if ((rc = check_ready(c))) return rc;
    const int order = g->b[0]->d.time_order;
    for (int step = 0; step < nsteps; step++) {
        for (shx_case *c : g->b)
            if ((rc = step_begin(c))) return rc;
        for (int s = 0; s < order; s++) {
            if ((rc = join_blocks(g)) || (rc = gather(g, false)) || (rc = fork_blocks(g))) return rc;
            for (shx_case *c : g->b)
                if ((rc = step_stage(c, s, tau, STEP_NAN))) return rc;
        }
        for (shx_case *c : g->b) step_end(c);
        int bad = 0;
        for (shx_case *c : g->b) {
            int fresh = 0;
            if ((rc = nan_found(c, fresh))) return rc;
            bad += fresh;
        }
        if (bad > 0)
            return set_err(SHX_ERR_NAN, "checkNAN: %d interior nodes with a non-finite density after step %d of %d "
                           "(set to 1e6)", bad, step + 1, nsteps);
    }
    if ((rc = join_blocks(g))) return rc;
    return SHX_OK;
}

// ---- batches of independent cases --------------------------------------------------------------
// A batch advances many cases of uneven size together.  Cases that share the kernel templates
// (dimension, scheme, metric kind, arithmetic form, viscosity, RK order) form a group; per stage
// every kernel class of a group is one launch over the concatenated tile lists of its cases
// (k_*_batch), and the launches of one full RK step of every group are captured once into a HIP
// graph that is replayed per step.  The step keeps each case's U_lastStep buffer in place: the
// last stage writes the new state over U_n pointwise (each node reads U_n before it is
// overwritten), so the captured pointers stay valid from step to step.  Blocks of a launch walk
// its work list with a grid stride; the number of resident blocks per class is chosen by
// shx_batch_tune.
struct BatchLaunch {
    const void *fn, *fnp;          // flat and persistent kernels; launched: fn when grid == total
    const void *run;
    int threads, total, grid, klass;
    int group;                     // kernel-template group (one lane of the step graph)
    size_t args_off, work_off;
    const void *A;
    const int4 *work;
};

enum { BK_GHOST, BK_VALUES, BK_GRAD, BK_WENO, BK_VISC, BK_PLANE, BK_NUM };

struct shx_batch {
    std::vector<shx_case *> cases;
    std::vector<double> tau;
    hipStream_t stream = nullptr;
    std::vector<BatchLaunch> seq;
    std::vector<char> host;      // argument tables, laid out as on the device
    char *dev = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipEvent_t done = nullptr;
    int factor[BK_NUM];          // resident blocks per CU per class (0: one block per work item)
    int ncu = 0;
    int use_graph = 1;           // 0: launch the step's kernels directly (SHX_BATCH_GRAPH=0)
    // Groups share no data, so every group runs on a lane stream of its own between a fork and a
    // join on `stream`: kernels of different groups (a memory-bound fill of one beside the sweeps
    // of another, the tail of one launch beside the head of the next) overlap on the device.
    int ngroups = 0, cur_group = 0;
    std::vector<hipStream_t> lanes;
    std::vector<hipEvent_t> joins;
    hipEvent_t fork = nullptr;
    // checkNAN fused into every case's last stage: running counts per case on the device, read by
    // shx_batch_synchronize into a pinned host copy; nan_seen: the counts already reported
    int *d_nan = nullptr, *h_nan = nullptr;
    std::vector<int> nan_seen;
};

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// stage buffers with the state kept in place: (in, out) per stage
static void batch_buffers(const shx_case *c, int s, int &in, int &out)
{
    const int cur = c->cur, bx = (cur + 1) % 3, by = (cur + 2) % 3;
    if (c->d.time_order == 4) {
        static const int io[4][2] = {{0, 1}, {1, 2}, {2, 1}, {1, 0}};
        const int map[3] = {cur, bx, by};
        in = map[io[s][0]]; out = map[io[s][1]];
    } else {
        static const int io[3][2] = {{0, 1}, {1, 2}, {2, 0}};
        const int map[3] = {cur, bx, by};
        in = map[io[s][0]]; out = map[io[s][1]];
    }
}

// append one launch over `cs` with per-case argument records `recs` (rsize bytes each) and grids
// Work-list order, as the single-case launches order their tiles (sweep_tile): ORDER_NODES keeps
// every case's blocks in x order; ORDER_SWEEP lists sweep tiles fastest and places them on the
// XCDs as xcd_order does.
enum { ORDER_NODES, ORDER_SWEEP };
static int host_xcd_order(const int p, const int total)
{
    const int per = total >> 3, rem = total & 7, x = p & 7, s = p >> 3;
    return x * per + std::min(x, rem) + s;
}
static void batch_add(shx_batch *b, const void *fn, const void *fnp, int threads, int klass,
                      const std::vector<char> &recs, size_t rsize, const std::vector<dim3> &grids,
                      int order = ORDER_NODES)
{
    BatchLaunch L;
    memset(&L, 0, sizeof L);
    L.fn = fn; L.fnp = fnp; L.threads = threads; L.klass = klass; L.group = b->cur_group;
    const int nc = (int)grids.size();
    std::vector<int4> tiles;
    for (int i = 0; i < nc; i++) {
        const dim3 g = grids[i];      // node-parallel kernels: (blocks, 1, 1)
        if (order == ORDER_SWEEP) {
            for (unsigned y = 0; y < g.y; y++)
                for (unsigned x = 0; x < g.x; x++)
                    for (unsigned z = 0; z < g.z; z++) tiles.push_back(make_int4(i, (int)x, (int)y, (int)z));
        } else {
            for (unsigned z = 0; z < g.z; z++)
                for (unsigned y = 0; y < g.y; y++)
                    for (unsigned x = 0; x < g.x; x++) tiles.push_back(make_int4(i, (int)x, (int)y, (int)z));
        }
    }
    std::vector<int4> work(tiles.size());
    const int nt = (int)tiles.size();
    for (int q = 0; q < nt; q++) work[q] = (order == ORDER_NODES) ? tiles[q] : tiles[host_xcd_order(q, nt)];
    L.total = (int)work.size();
    if (work.empty()) work.push_back(make_int4(0, 0, 0, 0));
    L.args_off = align256(b->host.size());
    b->host.resize(L.args_off + recs.size());
    memcpy(b->host.data() + L.args_off, recs.data(), recs.size());
    L.work_off = align256(b->host.size());
    b->host.resize(L.work_off + work.size() * sizeof(int4));
    memcpy(b->host.data() + L.work_off, work.data(), work.size() * sizeof(int4));
    (void)rsize;
    b->seq.push_back(L);
}

template <class T>
static void put(std::vector<char> &recs, const T &r)
{
    const size_t o = recs.size();
    recs.resize(o + sizeof(T));
    memcpy(recs.data() + o, &r, sizeof(T));
}

// the launches of one RK step of one group (cases with identical kernel templates)
static int batch_group(shx_batch *b, const std::vector<shx_case *> &g, const std::vector<double> &tau)
{
    shx_case *c0 = g[0];
    const int dims = c0->gm.dims, S = c0->d.space_order;
    const int nc = (int)g.size();
    for (int s = 0; s < c0->d.time_order; s++) {
        std::vector<RkArgs> rk(nc);
        std::vector<double *const *> in(nc), out(nc);
        for (int i = 0; i < nc; i++) {
            int ib, ob;
            batch_buffers(g[i], s, ib, ob);
            in[i] = g[i]->prim[ib];
            out[i] = g[i]->prim[ob];
            rk[i] = rk_args(g[i], g[i]->prim[ib], g[i]->prim[ob], s, tau[i]);
            if (s == c0->d.time_order - 1 && b->d_nan) {
                // checkNAN on the step's new state (as shx_run), counted per case
                const long k = std::find(b->cases.begin(), b->cases.end(), g[i]) - b->cases.begin();
                rk[i].nan_cnt = b->d_nan + k;
                rk[i].nanP = g[i]->P;
            }
        }
        if (s == 0) {   // start of the step: step-start ghost state of every Rudy face
            for (int f = 0; f < 2 * dims; f++) {
                std::vector<char> recs;
                std::vector<dim3> grids;
                long any = 0;
                for (int i = 0; i < nc; i++) {
                    BcArgs a;
                    long nodes;
                    face_args(g[i], in[i], f, tau[i], a, nodes);
                    if (g[i]->d.bc[f] != SHX_BC_OUTFLOW_RUDY) nodes = 0;
                    put(recs, a);
                    grids.push_back(dim3(nblk(nodes, 256)));
                    any += nodes;
                }
                if (any) batch_add(b, (const void *)&k_face_save_batch<false>, (const void *)&k_face_save_batch<true>, 256, BK_GHOST, recs, sizeof(BcArgs), grids);
            }
        }
        // cases that read ghosts at their image need none filled, but the state keeps those of the
        // step's start, as it always has in a batch
        auto fills = [&](const shx_case *c) { return s == 0 || !state_wraps(c); };
        if (c0->d.inviscid) {   // periodic ghost fill of the stage input
            std::vector<char> recs;
            std::vector<dim3> grids;
            long any = 0;
            for (int i = 0; i < nc; i++) {
                GhostArgs a;
                memset(&a, 0, sizeof a);
                for (int m = 0; m < 5; m++) a.f.f[m] = in[i][m];
                a.nf = 5; a.gm = g[i]->gm;
                put(recs, a);
                const long nodes = fills(g[i]) ? g[i]->gm.ntot : 0;
                grids.push_back(dim3(nblk(nodes, 256)));
                any += nodes;
            }
            if (any) batch_add(b, (const void *)&k_ghost_batch<false>, (const void *)&k_ghost_batch<true>, 256, BK_GHOST, recs, sizeof(GhostArgs), grids);
        }
        // face writers, one launch per face in the reference's order (after CalcValues when viscous);
        // a case contributes no blocks to the launch of a periodic face
        auto add_faces = [&]() {
            for (int f = 0; f < 2 * dims; f++) {
                std::vector<char> recs;
                std::vector<dim3> grids;
                long any = 0;
                for (int i = 0; i < nc; i++) {
                    BcArgs a;
                    long nodes;
                    face_args(g[i], in[i], f, tau[i], a, nodes);
                    put(recs, a);
                    grids.push_back(dim3(nblk(nodes, 256)));
                    any += nodes;
                }
                if (any) batch_add(b, (const void *)&k_face_batch<false>, (const void *)&k_face_batch<true>, 256, BK_GHOST, recs, sizeof(BcArgs), grids);
            }
        };
        if (c0->d.inviscid) {
            // stored p and c of the cases with subsonic outflow faces
            std::vector<char> recs;
            std::vector<dim3> grids;
            long any = 0;
            for (int i = 0; i < nc; i++) {
                ValuesArgs a;
                memset(&a, 0, sizeof a);
                for (int m = 0; m < 5; m++) a.pr.f[m] = in[i][m];
                a.P = g[i]->P; a.C = g[i]->C; a.gm = g[i]->gm; a.k = g[i]->k;
                put(recs, a);
                const long nodes = g[i]->pc ? g[i]->gm.ntot : 0;
                grids.push_back(dim3(nblk(nodes, 256)));
                any += nodes;
            }
            if (any) batch_add(b, (const void *)&k_values_batch<false>, (const void *)&k_values_batch<true>, 256, BK_VALUES, recs, sizeof(ValuesArgs), grids);
            add_faces();
        }
        if (!c0->d.inviscid) {
            // periodic ghost fill of the stage input with CalcValues
            std::vector<char> recs, grecs;
            std::vector<dim3> grids, ggrids;
            long cols = 0, any = 0;
            for (int i = 0; i < nc; i++) cols += march_columns(g[i]->gm, false);
            for (int i = 0; i < nc; i++) {
                shx_case *c = g[i];
                GhostValuesArgs a;
                memset(&a, 0, sizeof a);
                for (int m = 0; m < 5; m++) a.pr.f[m] = in[i][m];
                a.T = c->T; a.mu = c->mu; a.P = c->P; a.C = c->C; a.gm = c->gm; a.k = c->k;
                put(recs, a);
                const long nodes = fills(c) ? c->gm.ntot : 0;
                grids.push_back(dim3(nblk(nodes, 256)));
                any += nodes;
                if (dims == 2) continue;
                const int planes = march_planes(c, cols);
                put(grecs, grad_args(c, in[i], false, planes));
                ggrids.push_back(march_grid(c->gm, false, planes));
            }
            if (any) batch_add(b, (const void *)&k_ghost_values_batch<false>, (const void *)&k_ghost_values_batch<true>, 256, BK_VALUES, recs, sizeof(GhostValuesArgs), grids);
            add_faces();
            // the march with the viscous xi terms follows the WENO xi sweep (below)
            if (dims == 3 && !fuse_xi(c0))
                batch_add(b, march_kernel(S, !c0->diag, true, false), march_kernel(S, !c0->diag, true, true), GK * GJ,
                          BK_GRAD, grecs, sizeof(GradArgs), ggrids, ORDER_NODES);
        }
        if (dims == 2) {
            const Pick p = plane_pick(c0);
            std::vector<char> recs;
            std::vector<dim3> grids;
            for (int i = 0; i < nc; i++) {
                const PlaneArgs z = plane_args(g[i], in[i], &rk[i], state_wraps(g[i]));
                put(recs, z);
                grids.push_back(dim3(z.nt[0] * z.nt[1]));
            }
            batch_add(b, p.batch, p.batchp, 512, BK_PLANE, recs, sizeof(PlaneArgs), grids, ORDER_NODES);
        }
        // the same sweep sequence as stage_fluxes (fused eta and zeta directions where they apply)
        const bool fz = fuse_zeta(c0), fx = fuse_xi(c0), fe = fuse_eta(c0);
        const int nsep = dims == 2 ? 0 : (fz ? dims - 1 : dims);
        for (int dir = 0; dir < nsep; dir++) {
            if (fe && dir == 1) continue;
            const Pick p = weno_pick(c0, dir, dir == 2 ? zeta_tile(g.data(), nc) : c0->wtile[dir]);
            std::vector<char> recs;
            std::vector<dim3> grids;
            for (int i = 0; i < nc; i++) {
                const bool wrap = state_wraps(g[i]);
                const WenoArgs a = weno_args(g[i], in[i], dir, dir == 0, wrap);
                if (dir == 2) put(recs, weno_last_args(g[i], in[i], 0, c0->d.inviscid ? &rk[i] : nullptr, wrap));
                else put(recs, a);
                grids.push_back(sweep_grid(a.nA, a.oA, a.alignA, a.nB, a.nD, p));
            }
            batch_add(b, p.batch, p.batchp, p.TA * p.TDI, BK_WENO, recs, dir == 2 ? sizeof(WenoLastArgs) : sizeof(WenoArgs),
                      grids, ORDER_SWEEP);
        }
        if (fx) {
            std::vector<char> recs;
            std::vector<dim3> grids;
            long cols = 0;
            for (int i = 0; i < nc; i++) cols += march_columns(g[i]->gm, true);
            for (int i = 0; i < nc; i++) {
                const int planes = march_planes(g[i], cols);
                put(recs, grad_args(g[i], in[i], true, planes));
                grids.push_back(march_grid(g[i]->gm, true, planes));
            }
            batch_add(b, (const void *)&k_march_xi_batch<false>, (const void *)&k_march_xi_batch<true>, GKX * GJX,
                      BK_GRAD, recs, sizeof(GradArgs), grids, ORDER_NODES);
        }
        if (fz) {
            const Pick p = zeta_pick(c0, zeta_tile(g.data(), nc));
            std::vector<char> zrecs;
            std::vector<dim3> grids;
            // viscous xi (unless the march took it) and eta (or the fused eta kernel), then the
            // fused zeta kernel
            for (int dir = fx ? 1 : 0; dir < nsep; dir++) {
                if (fe && dir == 1) {
                    const Pick pe = eta_pick(c0);
                    std::vector<char> recs;
                    std::vector<dim3> eg;
                    for (int i = 0; i < nc; i++) {
                        const EtaArgs z = eta_args(g[i], in[i]);
                        put(recs, z);
                        eg.push_back(sweep_grid(z.w.nA, z.w.oA, z.w.alignA, z.w.nB, z.w.nD, pe));
                    }
                    batch_add(b, pe.batch, pe.batchp, pe.TA * pe.TDI, BK_VISC, recs, sizeof(EtaArgs), eg, ORDER_SWEEP);
                    continue;
                }
                const Pick pv = visc_pick(c0, dir);
                std::vector<char> recs;
                std::vector<dim3> vg;
                for (int i = 0; i < nc; i++) {
                    const ViscArgs a = visc_args(g[i], in[i], dir, nullptr);
                    put(recs, a);
                    vg.push_back(sweep_grid(a.nA, a.oA, a.alignA, a.nB, a.nD, pv));
                }
                batch_add(b, pv.batch, pv.batchp, pv.TA * pv.TDI, BK_VISC, recs, sizeof(ViscArgs), vg,
                          sweep_order(true, dir) ? ORDER_SWEEP : ORDER_NODES);
            }
            for (int i = 0; i < nc; i++) {
                const ZetaArgs z = zeta_args(g[i], in[i], &rk[i]);
                put(zrecs, z);
                grids.push_back(sweep_grid(z.w.nA, z.w.oA, z.w.alignA, z.w.nB, z.w.nD, p));
            }
            batch_add(b, p.batch, p.batchp, p.TA * p.TDI, BK_VISC, zrecs, sizeof(ZetaArgs), grids, ORDER_SWEEP);
        } else if (dims == 3 && !c0->d.inviscid) {
            for (int dir = 0; dir < dims; dir++) {
                const Pick p = visc_pick(c0, dir);
                std::vector<char> recs;
                std::vector<dim3> grids;
                for (int i = 0; i < nc; i++) {
                    const ViscArgs a = visc_args(g[i], in[i], dir, dir == dims - 1 ? &rk[i] : nullptr);
                    put(recs, a);
                    grids.push_back(sweep_grid(a.nA, a.oA, a.alignA, a.nB, a.nD, p));
                }
                batch_add(b, p.batch, p.batchp, p.TA * p.TDI, BK_VISC, recs, sizeof(ViscArgs), grids,
                          sweep_order(true, dir) ? ORDER_SWEEP : ORDER_NODES);
            }
        }
        {   // ghost layers of non-periodic directions into the next stage buffer (ghost nodes only,
            // so the in-place last stage, whose update writes interior nodes of U_n, is unaffected)
            std::vector<char> recs;
            std::vector<dim3> grids;
            long any = 0;
            for (int i = 0; i < nc; i++) {
                CarryArgs a;
                memset(&a, 0, sizeof a);
                for (int m = 0; m < 5; m++) { a.from.f[m] = in[i][m]; a.to.f[m] = out[i][m]; }
                a.gm = g[i]->gm;
                put(recs, a);
                const long nodes = g[i]->faces ? g[i]->gm.ntot : 0;
                grids.push_back(dim3(nblk(nodes, 256)));
                any += nodes;
            }
            if (any) batch_add(b, (const void *)&k_carry_batch<false>, (const void *)&k_carry_batch<true>, 256, BK_GHOST, recs, sizeof(CarryArgs), grids);
        }
    }
    return SHX_OK;
}

static bool same_group(const shx_case *a, const shx_case *c)
{
    return a->gm.dims == c->gm.dims && a->d.space_order == c->d.space_order && a->diag == c->diag &&
           a->d.precision == c->d.precision && a->d.inviscid == c->d.inviscid && a->d.time_order == c->d.time_order &&
           a->wtile[0] == c->wtile[0] && a->wtile[1] == c->wtile[1] && a->wtile[2] == c->wtile[2];
}

// (re)build the argument tables of every launch for the current time steps
static int batch_build(shx_batch *b)
{
    b->seq.clear();
    b->host.clear();
    b->ngroups = 0;
    std::vector<int> done(b->cases.size(), 0);
    for (size_t i = 0; i < b->cases.size(); i++) {
        if (done[i]) continue;
        std::vector<shx_case *> g;
        std::vector<double> t;
        for (size_t j = i; j < b->cases.size(); j++)
            if (!done[j] && same_group(b->cases[i], b->cases[j])) {
                g.push_back(b->cases[j]);
                t.push_back(b->tau[j]);
                done[j] = 1;
            }
        b->cur_group = b->ngroups++;
        int rc = batch_group(b, g, t);
        if (rc) return rc;
    }
    return SHX_OK;
}

static int batch_grids(shx_batch *b)
{
    for (BatchLaunch &L : b->seq) {
        const int f = b->factor[L.klass];
        if (f <= 0) { L.grid = std::max(L.total, 1); L.run = L.fn; continue; }
        int per = 0;
        HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, L.fnp, L.threads, 0));
        L.grid = std::max(1, std::min(L.total, std::max(1, per) * b->ncu * f));
        L.run = L.fnp;
    }
    return SHX_OK;
}

// lane streams and events for the current number of groups
static int batch_lanes(shx_batch *b)
{
    if (!b->fork) HIPCHK(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
    while ((int)b->lanes.size() < b->ngroups) {
        hipStream_t s;
        hipEvent_t e;
        HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        b->lanes.push_back(s);
        HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        b->joins.push_back(e);
    }
    return SHX_OK;
}

// one RK step of every group: fork from `stream`, each group's launches on its lane, join
static hipError_t batch_enqueue(shx_batch *b)
{
    const bool fan = b->ngroups > 1;
    hipError_t e = hipSuccess;
    if (fan) {
        e = hipEventRecord(b->fork, b->stream);
        for (int g = 0; g < b->ngroups && e == hipSuccess; g++) e = hipStreamWaitEvent(b->lanes[g], b->fork, 0);
    }
    for (BatchLaunch &L : b->seq) {
        if (e != hipSuccess) break;
        void *args[] = {&L.A, &L.work, &L.total};
        e = hipLaunchKernel(L.run, dim3(L.grid), dim3(L.threads), args, 0, fan ? b->lanes[L.group] : b->stream);
    }
    if (fan)
        for (int g = 0; g < b->ngroups && e == hipSuccess; g++) {
            e = hipEventRecord(b->joins[g], b->lanes[g]);
            if (e == hipSuccess) e = hipStreamWaitEvent(b->stream, b->joins[g], 0);
        }
    return e;
}

// (the graph before it stays until the new one is there)
static int batch_capture(shx_batch *b)
{
    int rc = batch_lanes(b);
    if (rc) return rc;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    hipError_t e = batch_enqueue(b);
    const hipError_t end = hipStreamEndCapture(b->stream, &graph);
    if (e == hipSuccess) e = end;
    if (e == hipSuccess) e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        if (graph) hipGraphDestroy(graph);
        return set_err(SHX_ERR_HIP, "batch capture: %s", hipGetErrorString(e));
    }
    if (b->exec) hipGraphExecDestroy(b->exec);
    if (b->graph) hipGraphDestroy(b->graph);
    b->graph = graph;
    b->exec = exec;
    return SHX_OK;
}

// upload the tables: into the device's own where their layout is the same, which keeps captured pointers
// valid, else into a new one (fresh)
static int batch_upload(shx_batch *b, bool fresh)
{
    if (fresh) {
        if (b->dev) hipFree(b->dev);
        b->dev = nullptr;
        HIPCHK(hipMalloc((void **)&b->dev, std::max<size_t>(b->host.size(), 256)));
    }
    HIPCHK(hipMemcpyAsync(b->dev, b->host.data(), b->host.size(), hipMemcpyHostToDevice, b->stream));
    for (BatchLaunch &L : b->seq) {
        L.A = b->dev + L.args_off;
        L.work = (const int4 *)(b->dev + L.work_off);
    }
    HIPCHK(hipStreamSynchronize(b->stream));
    return SHX_OK;
}

extern "C" int shx_batch_create(shx_case *const *cases, int ncases, const double *tau, shx_batch **out)
{
    if (!cases || !tau || !out || ncases <= 0) return set_err(SHX_ERR_ARG, "null argument or empty batch");
    *out = nullptr;
    for (int i = 0; i < ncases; i++) {
        shx_case *c = cases[i];
        int rc = check_ready(c);
        if (rc) return rc;
        if (!(tau[i] > 0.0)) return set_err(SHX_ERR_ARG, "case %d: tau must be positive", i);
        for (int j = 0; j < i; j++)
            if (cases[j] == c) return set_err(SHX_ERR_ARG, "case %d appears twice", i);
        if (c->batch) return set_err(SHX_ERR_STATE, "case %d is in another batch", i);
        if (c->iface) return set_err(SHX_ERR_UNSUPPORTED, "case %d has interface faces (a block of a multi-block case)", i);
        HIPCHK(hipStreamSynchronize(c->stream));
    }
    shx_batch *b = new shx_batch();
    b->cases.assign(cases, cases + ncases);
    b->tau.assign(tau, tau + ncases);
    for (int k = 0; k < BK_NUM; k++) b->factor[k] = 0;
    {
        const char *env = getenv("SHX_BATCH_GRAPH");
        if (env && env[0] == '0') b->use_graph = 0;
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&b->ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipStreamCreate(&b->stream);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b->done, hipEventDisableTiming);
    if (e == hipSuccess) e = hipMalloc((void **)&b->d_nan, sizeof(int) * (size_t)ncases);
    if (e == hipSuccess) e = hipHostMalloc((void **)&b->h_nan, sizeof(int) * (size_t)ncases, hipHostMallocDefault);
    if (e == hipSuccess) e = hipMemsetAsync(b->d_nan, 0, sizeof(int) * (size_t)ncases, b->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
    if (e != hipSuccess) { shx_batch_destroy(b); return set_err(SHX_ERR_HIP, "batch setup: %s", hipGetErrorString(e)); }
    b->nan_seen.assign((size_t)ncases, 0);
    int rc = batch_build(b);
    if (!rc) rc = batch_upload(b, true);
    if (!rc) rc = batch_grids(b);
    if (!rc) rc = batch_capture(b);
    if (rc) { shx_batch_destroy(b); return rc; }
    for (shx_case *c : b->cases) c->batch = b;
    *out = b;
    return SHX_OK;
}

// the launches of two builds read their tables at the same places with the same grids
static bool same_layout(const std::vector<BatchLaunch> &a, const std::vector<BatchLaunch> &b)
{
    if (a.size() != b.size()) return false;
    for (size_t i = 0; i < a.size(); i++)
        if (a[i].fn != b[i].fn || a[i].fnp != b[i].fnp || a[i].threads != b[i].threads || a[i].total != b[i].total ||
            a[i].klass != b[i].klass || a[i].group != b[i].group || a[i].args_off != b[i].args_off ||
            a[i].work_off != b[i].work_off)
            return false;
    return true;
}

// The cases can change under a batch what its launches are: post-processing makes a case keep its
// pressure (which adds passes, and ghost fills where it read ghosts at their image), a new metric or
// shx_tune its kernels.  A build that no longer fits the tables and the captured graph replaces both; if
// that fails, the batch stays as it was.
extern "C" int shx_batch_set_tau(shx_batch *b, const double *tau)
{
    if (!b || !tau) return set_err(SHX_ERR_ARG, "null argument");
    for (size_t i = 0; i < b->cases.size(); i++)
        if (!(tau[i] > 0.0)) return set_err(SHX_ERR_ARG, "case %zu: tau must be positive", i);
    HIPCHK(hipStreamSynchronize(b->stream));
    std::vector<BatchLaunch> seq;
    std::vector<char> host;
    std::vector<double> old_tau(tau, tau + b->cases.size());
    seq.swap(b->seq); host.swap(b->host); old_tau.swap(b->tau);
    char *const dev = b->dev;
    const int ngroups = b->ngroups;
    int rc = batch_build(b);
    if (!rc && same_layout(seq, b->seq) && host.size() == b->host.size()) {
        for (size_t i = 0; i < b->seq.size(); i++) { b->seq[i].grid = seq[i].grid; b->seq[i].run = seq[i].run; }
        return batch_upload(b, false);
    }
    b->dev = nullptr;
    if (!rc) rc = batch_upload(b, true);
    if (!rc) rc = batch_grids(b);
    if (!rc) rc = batch_capture(b);
    if (rc) {
        if (b->dev) hipFree(b->dev);
        b->dev = dev;
        b->seq.swap(seq); b->host.swap(host); b->tau.swap(old_tau);
        b->ngroups = ngroups;
        return rc;
    }
    hipFree(dev);
    return SHX_OK;
}

extern "C" int shx_batch_run(shx_batch *b, int nsteps)
{
    if (!b) return set_err(SHX_ERR_ARG, "null batch");
    if (nsteps < 0) return set_err(SHX_ERR_ARG, "negative step count");
    // order the batch after earlier work on every case's stream, and later work after the batch
    for (shx_case *c : b->cases) {
        HIPCHK(hipEventRecord(b->done, c->stream));
        HIPCHK(hipStreamWaitEvent(b->stream, b->done, 0));
    }
    for (int s = 0; s < nsteps; s++) {
        if (b->use_graph) {
            HIPCHK(hipGraphLaunch(b->exec, b->stream));
        } else {
            HIPCHK(batch_enqueue(b));
        }
    }
    HIPCHK(hipEventRecord(b->done, b->stream));
    for (shx_case *c : b->cases) HIPCHK(hipStreamWaitEvent(c->stream, b->done, 0));
    return SHX_OK;
}

// Waits for the batch, then reads the fused checkNAN counts: SHX_ERR_NAN names the cases whose
// new states held a non-finite density in the steps since the last call (those nodes hold 1e6).
static int batch_nan_read(shx_batch *b)
{
    const size_t n = b->cases.size();
    HIPCHK(hipMemcpyAsync(b->h_nan, b->d_nan, sizeof(int) * n, hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return SHX_OK;
}

extern "C" int shx_batch_synchronize(shx_batch *b)
{
    if (!b) return set_err(SHX_ERR_ARG, "null batch");
    int rc = batch_nan_read(b);
    if (rc) return rc;
    char msg[400];
    int len = 0, bad = 0;
    for (size_t i = 0; i < b->cases.size(); i++) {
        const int fresh = b->h_nan[i] - b->nan_seen[i];
        b->nan_seen[i] = b->h_nan[i];
        if (fresh <= 0) continue;
        if (bad++ < 8 && len < (int)sizeof msg - 64)
            len += snprintf(msg + len, sizeof msg - len, "%scase %zu: %d", bad > 1 ? ", " : "", i, fresh);
    }
    if (bad)
        return set_err(SHX_ERR_NAN, "checkNAN: interior nodes with a non-finite density (set to 1e6) in %d case%s "
                       "since the last synchronize (%s%s)", bad, bad > 1 ? "s" : "", msg, bad > 8 ? ", ..." : "");
    return SHX_OK;
}

extern "C" int shx_batch_nan_counts(shx_batch *b, int *counts)
{
    if (!b || !counts) return set_err(SHX_ERR_ARG, "null argument");
    int rc = batch_nan_read(b);
    if (rc) return rc;
    for (size_t i = 0; i < b->cases.size(); i++) counts[i] = b->h_nan[i];
    return SHX_OK;
}

// Autotuning: for each kernel class in turn, time whole replayed steps with each candidate number
// of resident blocks per CU (0 = one block per work item) and keep the fastest.  The case states
// are restored afterwards, so tuning leaves the solution unchanged.
extern "C" int shx_batch_tune(shx_batch *b, int steps, int factors_out[6])
{
    if (!b) return set_err(SHX_ERR_ARG, "null batch");
    if (steps <= 0) steps = 1;
    HIPCHK(hipStreamSynchronize(b->stream));
    // snapshot U_lastStep of every case
    std::vector<double *> snap;
    for (shx_case *c : b->cases) {
        HIPCHK(hipStreamSynchronize(c->stream));
        const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
        for (int m = 0; m < 5; m++) {
            double *p = nullptr;
            HIPCHK(hipMalloc((void **)&p, bytes));
            HIPCHK(hipMemcpyAsync(p, c->prim[c->cur][m], bytes, hipMemcpyDeviceToDevice, b->stream));
            snap.push_back(p);
        }
    }
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    static const int cand[4] = {1, 2, 4, 0};
    int rc = SHX_OK;
    for (int k = 0; k < BK_NUM && !rc; k++) {
        bool used = false;
        for (const BatchLaunch &L : b->seq) used |= (L.klass == k);
        if (!used) continue;
        float best = 1e30f;
        int bestf = b->factor[k];
        for (int ci = 0; ci < 4 && !rc; ci++) {
            b->factor[k] = cand[ci];
            if ((rc = batch_grids(b)) || (rc = batch_capture(b))) break;
            HIPCHK(hipGraphLaunch(b->exec, b->stream));      // warm-up
            HIPCHK(hipEventRecord(e0, b->stream));
            for (int s = 0; s < steps; s++) HIPCHK(hipGraphLaunch(b->exec, b->stream));
            HIPCHK(hipEventRecord(e1, b->stream));
            HIPCHK(hipEventSynchronize(e1));
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, e0, e1));
            if (ms < best) { best = ms; bestf = cand[ci]; }
        }
        b->factor[k] = bestf;
    }
    // restore the states
    size_t si = 0;
    for (shx_case *c : b->cases) {
        const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
        for (int m = 0; m < 5; m++, si++) {
            HIPCHK(hipMemcpyAsync(c->prim[c->cur][m], snap[si], bytes, hipMemcpyDeviceToDevice, b->stream));
        }
    }
    HIPCHK(hipStreamSynchronize(b->stream));
    for (double *p : snap) hipFree(p);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc) return rc;
    // the tuning steps are not part of the solution: their checkNAN counts are not reported
    if ((rc = batch_nan_read(b))) return rc;
    for (size_t i = 0; i < b->cases.size(); i++) b->nan_seen[i] = b->h_nan[i];
    if ((rc = batch_grids(b)) || (rc = batch_capture(b))) return rc;
    if (factors_out)
        for (int k = 0; k < BK_NUM; k++) factors_out[k] = b->factor[k];
    return SHX_OK;
}

extern "C" int shx_batch_destroy(shx_batch *b)
{
    if (!b) return SHX_OK;
    if (b->stream) hipStreamSynchronize(b->stream);
    if (b->exec) hipGraphExecDestroy(b->exec);
    if (b->graph) hipGraphDestroy(b->graph);
    if (b->dev) hipFree(b->dev);
    if (b->done) hipEventDestroy(b->done);
    for (hipStream_t l : b->lanes) { hipStreamSynchronize(l); hipStreamDestroy(l); }
    for (hipEvent_t e : b->joins) hipEventDestroy(e);
    if (b->fork) hipEventDestroy(b->fork);
    if (b->d_nan) hipFree(b->d_nan);
    if (b->h_nan) hipHostFree(b->h_nan);
    if (b->stream) hipStreamDestroy(b->stream);
    for (shx_case *c : b->cases)
        if (c->batch == b) c->batch = nullptr;
    delete b;
    return SHX_OK;
}

// Tile autotuning: for every direction, time `reps` WENO sweeps of the current state with each
// tile variant and keep the fastest.  The sweeps only write Q, which every stage recomputes, so
// the state is unchanged.
extern "C" int shx_tune(shx_case *c, int reps, int choice[3])
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (reps <= 0) reps = 3;
    double *const *pr = c->prim[c->cur];
    if (c->gm.dims == 2) {            // 2D stages run on k_plane's tile
        if (choice)
            for (int d = 0; d < 3; d++) choice[d] = std::max(c->wtile[d], 0);
        return SHX_OK;
    }
    if ((rc = ghost_fill(c, pr, 5))) return rc;
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    for (int dir = 0; dir < c->gm.dims && !rc; dir++) {
        if (dir == 2 && fuse_zeta(c)) continue;      // the fused kernel's tile stays by zeta_tile
        if (dir == 1 && fuse_eta(c)) { c->wtile[1] = 1; continue; }   // the fused eta kernel's 8 x 32 tile
        float best = 1e30f;
        int bestv = 0;
        for (int v = 0; v < NWTILE && !rc; v++) {
            c->wtile[dir] = v;
            if ((rc = weno_sweep(c, pr, dir, 1))) break;          // warm-up
            HIPCHK(hipEventRecord(e0, c->stream));
            for (int r = 0; r < reps && !rc; r++) rc = weno_sweep(c, pr, dir, 1);
            HIPCHK(hipEventRecord(e1, c->stream));
            HIPCHK(hipEventSynchronize(e1));
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, e0, e1));
            if (ms < best) { best = ms; bestv = v; }
        }
        c->wtile[dir] = bestv;
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc) return rc;
    if (choice)
        for (int d = 0; d < 3; d++) choice[d] = (d == 2) ? zeta_tile(&c, 1) : c->wtile[d];
    if (c->timing) drain_events(c);
    return SHX_OK;
}

extern "C" int shx_run(shx_case *c, double tau, int nsteps)
{
    if (nsteps < 0) return set_err(SHX_ERR_ARG, "negative step count");
    for (int s = 0; s < nsteps; s++) {
        int rc = step_rk(c, tau, STEP_NAN);
        if (rc) return rc;
        int bad = 0;
        if ((rc = nan_found(c, bad))) return rc;
        if (bad > 0)
            return set_err(SHX_ERR_NAN, "checkNAN: %d interior nodes with a non-finite density after step %d of %d "
                           "(set to 1e6)", bad, s + 1, nsteps);
        if (c->timing && c->ev_used > 4096) { rc = drain_events(c); if (rc) return rc; }
    }
    return SHX_OK;
}

// the maximum node CFL sum red_fetch left (stream synchronized)
static double red_max(shx_case *c)
{
    const unsigned long long mb = *(volatile unsigned long long *)&c->h_io->red;
    double mx;
    memcpy(&mx, &mb, sizeof mx);
    return mx;
}
static int red_clear(shx_case *c)
{
    HIPCHK(hipMemsetAsync(c->d_red, 0, sizeof(unsigned long long) * RED_SLOTS, c->stream));
    return SHX_OK;
}
// the slots' maximum into the host's word, and the slots cleared for the next reduction: one small
// launch where a step used to end in a fill and two copies
static int red_fetch(shx_case *c)
{
    k_red_report<<<1, RED_SLOTS, 0, c->stream>>>(c->d_red, &c->h_io->red);
    LAUNCH_CHECK();
    return SHX_OK;
}

extern "C" int shx_run_cfl(shx_case *c, double cfl, int nsteps, double *time)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (nsteps < 0 || !(cfl > 0.0)) return set_err(SHX_ERR_ARG, "negative step count or bad cfl");
    if (c->rudy) return set_err(SHX_ERR_UNSUPPORTED, "CFL stepping with Rudy outflow faces (their relaxation uses tau)");
    const Geom &gm = c->gm;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    // the first step's maximum from the current state; later ones from the fused reduction
    CFields5 pf;
    CFields10 mf;
    for (int m = 0; m < 5; m++) pf.f[m] = c->prim[c->cur][m];
    for (int m = 0; m < 10; m++) mf.f[m] = c->met[m];
    if ((rc = red_clear(c))) return rc;
    if ((rc = tbeg(c, KT_REDUCE))) return rc;
    k_cfl_max<<<nblk(nint, 256), 256, 0, c->stream>>>(pf, mf, gm, c->k, c->d_red);
    LAUNCH_CHECK();
    if ((rc = tend(c))) return rc;
    if ((rc = red_fetch(c))) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    double t = 0.0;
    for (int s = 0; s < nsteps; s++) {
        const double mx = red_max(c);
        if (!(mx > 0.0) || !std::isfinite(mx)) return set_err(SHX_ERR_NAN, "CFL maximum %g before step %d", mx, s + 1);
        const double dt = cfl / mx;
        if ((rc = step_rk(c, dt, STEP_NAN | STEP_CFL))) return rc;
        if ((rc = red_fetch(c))) return rc;
        int bad = 0;
        if ((rc = nan_found(c, bad))) return rc;
        t += dt;
        if (time) *time = t;
        if (bad > 0)
            return set_err(SHX_ERR_NAN, "checkNAN: %d interior nodes with a non-finite density after step %d of %d "
                           "(set to 1e6)", bad, s + 1, nsteps);
        if (c->timing && c->ev_used > 4096) { rc = drain_events(c); if (rc) return rc; }
    }
    if (time) *time = t;
    return SHX_OK;
}

// The stored pressure of U_lastStep (the last stage's CalcValues value, which the RK update does
// not renew) is what the reference's post-processing reads.  Cases with subsonic outflow or slip
// wall faces keep it anyway; others start keeping it here, from the current state's own p.
static int keep_pressure(shx_case *c)
{
    if (c->pc) return SHX_OK;
    const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
    HIPCHK(hipMalloc((void **)&c->P, bytes));
    HIPCHK(hipMalloc((void **)&c->C, bytes));
    CFields5 cp;
    for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
    k_calc_values<<<nblk(c->gm.ntot, 256), 256, 0, c->stream>>>(cp, nullptr, nullptr, c->P, c->C, c->gm, c->k);
    LAUNCH_CHECK();
    c->pc = 1;
    return SHX_OK;
}

// U_lastStep's ghosts in the reference are those of the last stage's input (filled at that stage's
// start); the state buffer gets them before it is read whole (post-processing, backups).  The next
// step refills the periodic ghosts and carries the others, so stepping is unaffected.
static int sync_ghosts(shx_case *c)
{
    if (c->last_in < 0 || c->last_in == c->cur) return SHX_OK;
    CFields5 a;
    Fields5 b;
    for (int m = 0; m < 5; m++) { a.f[m] = c->prim[c->last_in][m]; b.f[m] = c->prim[c->cur][m]; }
    k_copy_ghosts<<<nblk(c->gm.ntot, 256), 256, 0, c->stream>>>(a, b, c->gm, ((c->gm.dims == 2 || c->d.inviscid) && !c->faces) ? 1 : 0);
    LAUNCH_CHECK();
    c->last_in = -1;
    return SHX_OK;
}

static int post_compute(shx_case *c)
{
    int rc = keep_pressure(c);
    if (rc) return rc;
    if ((rc = sync_ghosts(c))) return rc;
    const Geom &gm = c->gm;
    const size_t bytes = sizeof(double) * (size_t)gm.nalloc;
    for (int m = 0; m < 3; m++)
        if (!c->post[m]) {
            HIPCHK(hipMalloc((void **)&c->post[m], bytes));
            HIPCHK(hipMemsetAsync(c->post[m], 0, bytes, c->stream));
        }
    CFields5 cp;
    CFields10 mf;
    Fields5 out;
    memset(&out, 0, sizeof out);
    for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
    for (int m = 0; m < 10; m++) mf.f[m] = c->met[m];
    for (int m = 0; m < 3; m++) out.f[m] = c->post[m];
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    k_post<<<nblk(nint, 256), 256, 0, c->stream>>>(cp, c->P, mf, out, gm, c->k, c->d.space_order);
    LAUNCH_CHECK();
    return SHX_OK;
}

extern "C" int shx_post(shx_case *c, double *const out[3])
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!out) return set_err(SHX_ERR_ARG, "null output");
    if ((rc = post_compute(c))) return rc;
    for (int m = 0; m < 3; m++)
        if (out[m]) { rc = copy_out(c, out[m], c->post[m]); if (rc) return rc; }
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_film_open(shx_case *c, int samples)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (samples < 1) return set_err(SHX_ERR_ARG, "samples must be positive");
    if ((rc = keep_pressure(c))) return rc;
    const long nint = (long)c->gm.n[0] * c->gm.n[1] * c->gm.n[2];
    hipFree(c->film);
    c->film = nullptr;
    HIPCHK(hipMalloc((void **)&c->film, sizeof(double) * (size_t)8 * nint * samples));
    c->film_cap = samples;
    c->film_n = 0;
    c->film_time.assign(samples, 0.0);
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

// one sample of the current state into the film (CalcValuesForPost + WriteValuesFromUToFilm)
static int film_sample(shx_case *c, double time)
{
    if (c->film_n >= c->film_cap) return set_err(SHX_ERR_STATE, "film full (%d samples)", c->film_cap);
    int rc = post_compute(c);
    if (rc) return rc;
    const Geom &gm = c->gm;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    CFields5 cp, po;
    memset(&po, 0, sizeof po);
    for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
    for (int m = 0; m < 3; m++) po.f[m] = c->post[m];
    k_film<<<nblk(nint, 256), 256, 0, c->stream>>>(cp, c->P, po, c->film, nint, c->film_n, gm);
    LAUNCH_CHECK();
    c->film_time[c->film_n++] = time;
    return SHX_OK;
}

extern "C" int shx_film_sample(shx_case *c, double time)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!c->film) return set_err(SHX_ERR_STATE, "no film: call shx_film_open");
    return film_sample(c, time);
}

extern "C" int shx_film_download(shx_case *c, int sample, double *const out[8], double *time)
{
    if (!c || !out) return set_err(SHX_ERR_ARG, "null argument");
    if (!c->film || sample < 0 || sample >= c->film_n) return set_err(SHX_ERR_ARG, "no such sample");
    const long nint = (long)c->gm.n[0] * c->gm.n[1] * c->gm.n[2];
    for (int m = 0; m < 8; m++)
        if (out[m])
            HIPCHK(hipMemcpyAsync(out[m], c->film + ((long)sample * 8 + m) * nint, sizeof(double) * nint,
                                  hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (time) *time = c->film_time[sample];
    return SHX_OK;
}

extern "C" int shx_history_download(shx_case *c, double *time, double *p, double *u, double *v, double *w)
{
    if (!c) return set_err(SHX_ERR_ARG, "null argument");
    if (!c->hist) return set_err(SHX_ERR_STATE, "no probe history: run shx_simulate with probes");
    const size_t fs = sizeof(double) * (size_t)c->hist_np * c->hist_iters;
    double *out[4] = {p, u, v, w};
    for (int m = 0; m < 4; m++)
        if (out[m]) HIPCHK(hipMemcpyAsync(out[m], c->hist + (size_t)m * c->hist_np * c->hist_iters, fs,
                                          hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (time) memcpy(time, c->hist_time.data(), sizeof(double) * c->hist_iters);
    return SHX_OK;
}

extern "C" int shx_mms_error(shx_case *c, double out[4])
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!out) return set_err(SHX_ERR_ARG, "null output");
    if (!c->has_bs) return set_err(SHX_ERR_STATE, "no exact state: call shx_upload_boundary_state");
    if ((rc = keep_pressure(c))) return rc;
    const Geom &gm = c->gm;
    const long nplane = (long)gm.n[0] * gm.n[1];
    const int nb = (int)nblk(nplane, 256);
    double *part = nullptr, *dout = nullptr;
    HIPCHK(hipMalloc((void **)&part, sizeof(double) * 4 * (size_t)nb));
    HIPCHK(hipMalloc((void **)&dout, sizeof(double) * 4));
    CFields5 cp;
    for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
    const double N = (double)gm.n[0] * gm.n[1] * gm.n[2];
    k_mms_error<<<nb, 256, 0, c->stream>>>(cp, c->P, c->bs[0], c->bs[5], gm, N, part);
    LAUNCH_CHECK();
    k_mms_error_total<<<1, 256, 0, c->stream>>>(part, nb, dout);
    LAUNCH_CHECK();
    HIPCHK(hipMemcpyAsync(out, dout, sizeof(double) * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    hipFree(part);
    hipFree(dout);
    return SHX_OK;
}

// ---- the entry point that allocates nothing -------------------------------------------------
// shx_mms_error_static: shx_mms_error with its partial sums and result in a file-scope device
// array instead of per-call allocations, for callers that cannot allocate (code under HIP graph
// capture, serving loops).  Every call on a device shares that device's array: calls that overlap
// on one device race.  No element needs clearing: k_mms_error writes every partial it later sums
// and k_mms_error_total writes every result.
constexpr int SCRATCH_BLOCKS = 4096;                   // n0 * n1 <= SCRATCH_BLOCKS * 256 interior nodes
static __device__ __align__(256) double scratch[4 + 4 * SCRATCH_BLOCKS];
constexpr int MAX_DEVICES = 64;
static double *g_scratch[MAX_DEVICES];                 // scratch's address on each device

// scratch's device address on the case's device, looked up once per device with that device
// current (in host code the array's name is only a stand-in for the symbol)
static int scratch_ptr(const shx_case *c, double **ptr)
{
    if (c->dev < 0 || c->dev >= MAX_DEVICES) return set_err(SHX_ERR_UNSUPPORTED, "device %d", c->dev);
    if (!g_scratch[c->dev]) {
        int cur = 0;
        HIPCHK(hipGetDevice(&cur));
        if (cur != c->dev) HIPCHK(hipSetDevice(c->dev));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != c->dev) HIPCHK(hipSetDevice(cur));
        if (e != hipSuccess || !p) return set_err(SHX_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch[c->dev] = (double *)p;
    }
    *ptr = g_scratch[c->dev];
    return SHX_OK;
}

extern "C" int shx_mms_error_static(shx_case *c, double out[4])
{
    if (!c || !out) return set_err(SHX_ERR_ARG, "null argument");
    const Geom &gm = c->gm;
    const long nplane = (long)gm.n[0] * gm.n[1];
    const long nb = (long)nblk(nplane, 256);
    if (nb > SCRATCH_BLOCKS)
        return set_err(SHX_ERR_ARG, "shx_mms_error_static: n0 * n1 = %ld interior nodes per k plane exceeds the "
                       "static scratch (at most %d)", nplane, SCRATCH_BLOCKS * 256);
    int rc = check_ready(c);
    if (rc) return rc;
    if (!c->has_bs) return set_err(SHX_ERR_STATE, "no exact state: call shx_upload_boundary_state");
    if (!c->pc)
        return set_err(SHX_ERR_STATE, "shx_mms_error_static reads the stored pressure, which this case does not "
                       "keep yet (keeping it allocates): call shx_mms_error, shx_post or shx_film_open once first");
    double *scr = nullptr;
    if ((rc = scratch_ptr(c, &scr))) return rc;
    double *const dout = scr, *const part = scr + 4;
    CFields5 cp;
    for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
    const double N = (double)gm.n[0] * gm.n[1] * gm.n[2];
    k_mms_error<<<(unsigned)nb, 256, 0, c->stream>>>(cp, c->P, c->bs[0], c->bs[5], gm, N, part);
    LAUNCH_CHECK();
    k_mms_error_total<<<1, 256, 0, c->stream>>>(part, (int)nb, dout);
    LAUNCH_CHECK();
    HIPCHK(hipMemcpyAsync(c->h_io->mms, dout, sizeof(double) * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    for (int m = 0; m < 4; m++) out[m] = c->h_io->mms[m];
    return SHX_OK;
}

extern "C" int shx_film_count(const shx_case *c, int *count)
{
    if (!c || !count) return set_err(SHX_ERR_ARG, "null argument");
    *count = c->film_n;
    return SHX_OK;
}

// state (and stored p) of the case into / out of backup slot b (WriteValuesFromU1ToU2,
// src/Functions.c:2484-2508: every padded node); a reload writes every stage buffer, as an upload does
static int backup_io(shx_case *c, int b, bool save)
{
    const size_t bytes = sizeof(double) * (size_t)c->gm.nalloc;
    if (save) { int rc = sync_ghosts(c); if (rc) return rc; }
    if (!c->bk[b][0])
        for (int m = 0; m < 5; m++) HIPCHK(hipMalloc((void **)&c->bk[b][m], bytes));
    if (c->pc && !c->bkP[b]) HIPCHK(hipMalloc((void **)&c->bkP[b], bytes));
    for (int m = 0; m < 5; m++) {
        if (save) {
            HIPCHK(hipMemcpyAsync(c->bk[b][m], c->prim[c->cur][m], bytes, hipMemcpyDeviceToDevice, c->stream));
        } else {
            for (int s = 0; s < 3; s++)
                HIPCHK(hipMemcpyAsync(c->prim[s][m], c->bk[b][m], bytes, hipMemcpyDeviceToDevice, c->stream));
        }
    }
    if (c->pc) {
        if (save) HIPCHK(hipMemcpyAsync(c->bkP[b], c->P, bytes, hipMemcpyDeviceToDevice, c->stream));
        else HIPCHK(hipMemcpyAsync(c->P, c->bkP[b], bytes, hipMemcpyDeviceToDevice, c->stream));
    }
    if (!save) c->last_in = -1;
    return SHX_OK;
}

extern "C" int shx_simulate(shx_case *c, const shx_sim *sim, shx_sim_report *rep)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!sim || !rep) return set_err(SHX_ERR_ARG, "null argument");
    if (!(sim->tau > 0.0) || !(sim->L0 > 0.0) || !(sim->u0 > 0.0) || sim->end_iteration < sim->start_iteration ||
        sim->distance_backward < 1 || sim->number_resets < 0 || !(sim->decel_factor > 0.0) ||
        (sim->accelerator && !(sim->accel_factor > 0.0)))
        return set_err(SHX_ERR_ARG, "bad simulation parameters");
    const bool sampling = sim->samples > 0;
    if (sampling && (sim->iterations_between_samples < 1 || !c->film || c->film_cap < sim->samples))
        return set_err(SHX_ERR_ARG, "sampling needs iterations_between_samples >= 1 and a film of that many samples");
    if (sim->nprobes < 0 || (sim->nprobes > 0 && !sim->probes)) return set_err(SHX_ERR_ARG, "bad probe list");
    const Geom &gm = c->gm;
    // probes are the reference's linear indices (i ng1 ng2 + j ng2 + k); the device arrays use
    // padded row pitches
    std::vector<long> dev_probes(sim->nprobes);
    for (int q = 0; q < sim->nprobes; q++) {
        const long n = sim->probes[q];
        if (n < 0 || n >= gm.ntot) return set_err(SHX_ERR_ARG, "probe %d outside the grid", q);
        const int ijk[3] = {(int)(n / ((long)gm.ng[1] * gm.ng[2])), (int)((n / gm.ng[2]) % gm.ng[1]), (int)(n % gm.ng[2])};
        for (int d = 0; d < gm.dims; d++)
            if (ijk[d] < gm.lo[d] || ijk[d] >= gm.lo[d] + gm.n[d]) return set_err(SHX_ERR_ARG, "probe %d is not an interior node", q);
        dev_probes[q] = (long)ijk[0] * gm.st[0] + (long)ijk[1] * gm.st[1] + (long)ijk[2] * gm.st[2];
    }
    memset(rep, 0, sizeof *rep);
    if ((sampling || sim->nprobes > 0) && (rc = keep_pressure(c))) return rc;
    const int iters = sim->end_iteration - sim->start_iteration;
    if (sim->nprobes > 0) {
        hipFree(c->d_probes); hipFree(c->hist);
        c->d_probes = nullptr; c->hist = nullptr;
        HIPCHK(hipMalloc((void **)&c->d_probes, sizeof(long) * sim->nprobes));
        HIPCHK(hipMemcpy(c->d_probes, dev_probes.data(), sizeof(long) * sim->nprobes, hipMemcpyHostToDevice));
        if (iters > 0) {
            HIPCHK(hipMalloc((void **)&c->hist, sizeof(double) * 4 * (size_t)sim->nprobes * iters));
            HIPCHK(hipMemsetAsync(c->hist, 0, sizeof(double) * 4 * (size_t)sim->nprobes * iters, c->stream));
        }
        c->hist_np = sim->nprobes;
        c->hist_iters = iters;
        c->hist_time.assign(iters, 0.0);
    }
    const double tau_start = sim->tau, L0 = sim->L0, u0 = sim->u0;
    const int end = sim->end_iteration, dback = sim->distance_backward, dnan = sim->distance_nan;
    double tau = tau_start, time = sim->time, last = sim->time_last_action;
    int dfwd = sim->distance_forward;
    // slot 0 is the reference's backup1, slot 1 its backup2 (src/SHOCK.c:531-540)
    int it_b[2] = {1, 999999};
    double time_b[2] = {time, 0.0};
    // sampling counters (int_iterationCounterSamples, int_actualSample) and their backups
    int counter = 0, sample = c->film_n;
    int counter_b[2] = {0, 0}, sample_b[2] = {sample, 0};
    if ((rc = backup_io(c, 0, true))) return rc;
    int last_run = sim->start_iteration;
    for (int it = sim->start_iteration + 1; it <= end; it++) {
        last_run = it;
        time += tau * L0 / u0;
        if ((rc = step_rk(c, tau, STEP_NAN))) return rc;
        int bad = 0;
        if ((rc = nan_found(c, bad))) return rc;
        if (bad > 0) {
            rep->nan_steps++;
            if (rep->resets >= sim->number_resets) { rep->aborted = 1; break; }
            rep->resets++;
            tau *= sim->decel_factor;
            dfwd = sim->distance_forward;
            const int b = (it_b[0] < it_b[1]) ? 0 : 1;
            if ((rc = backup_io(c, b, false))) return rc;
            last = time;
            time = time_b[b];
            it = it_b[b];
            sample = sample_b[b];
            counter = counter_b[b];
        } else if ((time - last) > dnan * tau * L0 / u0 && sim->accelerator && it + dback < end && tau < tau_start) {
            dfwd = sim->distance_forward;
            tau = tau_start;
            last = time;
            rep->tau_resets++;
        } else if ((time - last) > dfwd * tau * L0 / u0 && sim->accelerator && it + dback < end && tau >= tau_start) {
            dfwd = (int)(dfwd * 4.);
            tau *= sim->accel_factor;
            last = time;
            rep->accelerations++;
        }
        if (it % dback == 0) {
            if ((rc = backup_io(c, 0, true))) return rc;
            time_b[0] = time; it_b[0] = it; sample_b[0] = sample; counter_b[0] = counter;
        } else if ((it + dback / 2) % dback == 0) {
            if ((rc = backup_io(c, 1, true))) return rc;
            time_b[1] = time; it_b[1] = it; sample_b[1] = sample; counter_b[1] = counter;
        }
        // sampling (src/SHOCK.c:694-717): every iterations_between_samples iterations, from
        // start_sampling on, while samples remain; a rollback rewinds the sample index
        counter++;
        if (sampling && counter % sim->iterations_between_samples == 0 && sample < sim->samples &&
            it >= sim->start_sampling) {
            c->film_n = sample;
            if ((rc = film_sample(c, time))) return rc;
            sample++;
        }
        // history row of this iteration (src/Functions.c:5381-5417 index the history by
        // iteration - (start + 1)); a rollback to a backup older than the start (the first backup
        // is iteration 1 whatever the start, src/SHOCK.c:531-540) gives iterations before the
        // first row, which the reference writes out of bounds: they are not recorded here
        const int row = it - (sim->start_iteration + 1);
        if (sim->nprobes > 0 && row >= 0 && row < iters) {
            CFields5 cp;
            for (int m = 0; m < 5; m++) cp.f[m] = c->prim[c->cur][m];
            k_probe<<<nblk(sim->nprobes, 64), 64, 0, c->stream>>>(cp, c->P, c->d_probes, sim->nprobes, c->hist, row, iters);
            LAUNCH_CHECK();
            c->hist_time[row] = time;
        }
        if (c->timing && c->ev_used > 4096) { rc = drain_events(c); if (rc) return rc; }
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    rep->iteration = last_run;
    rep->time = time;
    rep->tau = tau;
    if (sampling) c->film_n = sample;
    rep->samples = sampling ? sample : c->film_n;
    return SHX_OK;
}

extern "C" int shx_rhs(shx_case *c, double *const q[5])
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!q) return set_err(SHX_ERR_ARG, "null output");
    if (c->iface) return set_err(SHX_ERR_UNSUPPORTED, "the case has interface faces (its ghosts need its multi-block case)");
    const Geom &gm = c->gm;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    // a Rudy face takes the current state as its step-start state, with tau = 0
    if ((rc = rudy_save(c, c->prim[c->cur]))) return rc;
    if ((rc = stage_fluxes(c, c->prim[c->cur], nullptr, 0.0))) return rc;
    if (c->has_src) {
        Fields5 qf;
        CFields5 sf;
        for (int m = 0; m < 5; m++) { qf.f[m] = c->q[m]; sf.f[m] = c->src[m]; }
        k_add_source<<<nblk(nint, 256), 256, 0, c->stream>>>(qf, sf, c->met[9], gm);
        LAUNCH_CHECK();
    }
    if ((rc = transfer(c, false, 5, c->q, q))) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_check_metric(shx_case *c, int *negative)
{
    if (!c || !negative) return set_err(SHX_ERR_ARG, "null argument");
    if (!c->has_metric) return set_err(SHX_ERR_STATE, "no metric yet");
    HIPCHK(hipMemsetAsync(c->d_cnt, 0, sizeof(int), c->stream));
    k_check_metric<<<nblk(c->gm.ntot, 256), 256, 0, c->stream>>>(c->met[9], c->gm, c->d_cnt);
    LAUNCH_CHECK();
    HIPCHK(hipMemcpyAsync(negative, c->d_cnt, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_check_nan(shx_case *c, int *count)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!count) return set_err(SHX_ERR_ARG, "null output");
    const Geom &gm = c->gm;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    Fields5 pf;
    for (int m = 0; m < 5; m++) pf.f[m] = c->prim[c->cur][m];
    HIPCHK(hipMemsetAsync(c->d_cnt, 0, sizeof(int), c->stream));
    if ((rc = tbeg(c, KT_REDUCE))) return rc;
    k_check_nan<<<nblk(nint, 256), 256, 0, c->stream>>>(pf, c->P, gm, c->d_cnt);
    LAUNCH_CHECK();
    if ((rc = tend(c))) return rc;
    HIPCHK(hipMemcpyAsync(count, c->d_cnt, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_cfl_dt(shx_case *c, double cfl, double *dt)
{
    int rc = check_ready(c);
    if (rc) return rc;
    if (!dt || !(cfl > 0.0)) return set_err(SHX_ERR_ARG, "bad cfl or null output");
    const Geom &gm = c->gm;
    const long nint = (long)gm.n[0] * gm.n[1] * gm.n[2];
    CFields5 pf;
    CFields10 mf;
    for (int m = 0; m < 5; m++) pf.f[m] = c->prim[c->cur][m];
    for (int m = 0; m < 10; m++) mf.f[m] = c->met[m];
    if ((rc = red_clear(c))) return rc;
    if ((rc = tbeg(c, KT_REDUCE))) return rc;
    k_cfl_max<<<nblk(nint, 256), 256, 0, c->stream>>>(pf, mf, gm, c->k, c->d_red);
    LAUNCH_CHECK();
    if ((rc = tend(c))) return rc;
    if ((rc = red_fetch(c))) return rc;
    HIPCHK(hipStreamSynchronize(c->stream));
    const double mx = red_max(c);
    *dt = mx > 0.0 ? cfl / mx : 0.0;
    return SHX_OK;
}

extern "C" int shx_copy_probe(shx_case *c, int reps)
{
    if (!c || reps < 0) return set_err(SHX_ERR_ARG, "bad argument");
    for (int r = 0; r < reps; r++) {
        k_copy<<<nblk(c->gm.nalloc, 256), 256, 0, c->stream>>>(c->T, c->mu, c->gm.nalloc);
        LAUNCH_CHECK();
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_synchronize(shx_case *c)
{
    if (!c) return set_err(SHX_ERR_ARG, "null handle");
    HIPCHK(hipStreamSynchronize(c->stream));
    return SHX_OK;
}

extern "C" int shx_set_timing(shx_case *c, int enable)
{
    if (!c) return set_err(SHX_ERR_ARG, "null handle");
    int rc = drain_events(c);
    if (rc) return rc;
    c->timing = enable ? 1 : 0;
    for (int s = 0; s < SHX_NUM_KERNELS; s++) { c->kt_ms[s] = 0.0; c->kt_n[s] = 0; }
    return SHX_OK;
}

extern "C" int shx_kernel_times(shx_case *c, const char *names[SHX_NUM_KERNELS], double ms[SHX_NUM_KERNELS],
                                int launches[SHX_NUM_KERNELS])
{
    if (!c) return set_err(SHX_ERR_ARG, "null handle");
    int rc = drain_events(c);
    if (rc) return rc;
    for (int s = 0; s < SHX_NUM_KERNELS; s++) {
        if (names) names[s] = g_knames[s];
        if (ms) ms[s] = c->kt_ms[s];
        if (launches) launches[s] = c->kt_n[s];
    }
    return SHX_OK;
}
