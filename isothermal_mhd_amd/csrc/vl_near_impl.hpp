// Fused FP64 stages whose faces read near neighbours only: the predictor (vanleer_mod.f90:
// 429-533) and the PLM corrector (:536-938), each with the upwind corner EMFs (:1884-2076)
// and the conservative + CT update (:2080-2259) in one launch, as k_vl_stage does for the
// other stages, with the same tiles, z-segments, masks and per-value arithmetic.
//
// What bounds them is the arithmetic of the solvers, whose divisions and square roots are
// two thirds of it, at two waves per SIMD (HLLD takes about 150 registers beside the march's
// 70; held to 168 registers for three waves, 90 to 240 of them spill: predictor 0.72 -> 0.94
// ms, corrector 0.95 -> 1.35).  So nothing is formed twice that the reference's arithmetic
// does not need twice:
//   - predictor: a cell's velocities are divided once and shared by its faces (and by the
//     centre EMFs) instead of once per face and side;
//   - corrector: a cell's primitives and its slope towards each axis are formed once (one
//     division instead of twelve);
//   - plane k+1 is in LDS (the corrector's with one ring cell on every side); x-neighbours'
//     states, and what else only x-neighbours read, come by lane shift; a plane's upper z-state
//     is carried to the next plane's face;
//   - everything of plane k+2 is loaded at the start of the pass that solves plane k+1.
// HLLD at 190 x 161 x 147, against the per-face form (k_vl_stage) over the same ranges: predictor
// 0.72 -> 0.655 ms, corrector 0.98 -> 0.945; in one round of segments 0.61 and 0.89.  The VALU is
// busy in 60 % of the cycles.  Not for the PLM corrector with the Roe solver (vs_near).
// Per plane k of the march:
//   A  the y- and x-faces of plane k+1 and the z-face k+1/2
//   D  corner EMFs of index k; plane k+2 replaces plane k+1 in LDS, its centre values are formed
//   G  update of plane k
// with a barrier after A and D.
#pragma once
#include "vl_stage_impl.hpp"

namespace imhd {

// Flux of a face from its two states (six rotated slots each): conserved values with their
// velocities vl, vr (predictor, flux_pred_calc's arithmetic) or interface primitives (corrector)
template <int RS, bool PRED>
__device__ __forceinline__ double near_solve(const double* sl, const double* sr, const double* vl, const double* vr,
                                             double wb, double cs, double* F) {
    if constexpr (PRED) {
        const double uL[7] = {sl[0], sl[1], sl[2], sl[3], wb, sl[4], sl[5]};
        const double uR[7] = {sr[0], sr[1], sr[2], sr[3], wb, sr[4], sr[5]};
        double smax = 0.0;
        if constexpr (RS == RS_HLLD) hlld<double, true>(uL, uR, cs * cs, F, smax, vl, vr);
        else if constexpr (RS == RS_HLLE) hlle<double, true>(uL, uR, cs * cs, F, smax, vl, vr);
        else riemann<RS>(uL, uR, cs, F, smax);
        return smax;
    } else {
        return plm_solve<double, RS>(sl, sr, wb, cs, F);
    }
}

template <int RS, bool PRED, int TX, int TY>
__global__ __launch_bounds__(TX * TY, 2) void k_vl_near(const BoxDesc* __restrict__ boxes, TilePlan plan,
                                                                StageArgs<double> a) {
    constexpr int N = TX * TY, RING = PRED ? 0 : 1, PX = TX + 2 * RING, PY = TY + 2 * RING, NR = 2 * (TX + TY);
    static_assert(64 % TX == 0 && NR <= N, "tile shape");
    // plane k+1, global order: the predictor's conserved values, the corrector's primitives
    // with one ring cell
    __shared__ double sW[7][PY * PX];
    __shared__ double sV[PRED ? 3 : 1][PRED ? N : 1];   // predictor: the velocities of plane k+1
    __shared__ double sF[4][N];        // y-face fluxes of plane k+1, global order
    __shared__ double sEf[2][N];       // [plane parity] x face E(2,0)
    __shared__ double sEz3[N];         // z face k+1/2: E(0,1)
    __shared__ double sC[2][3][N];     // [plane parity] centre Ex, Ez, m_y/rho
    __shared__ double sEz[N];          // corner Ez of plane k
    __shared__ double sEx[2][N];       // [index parity] corner Ex

    const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
    int b = 0;
    if (plan.nbox > 1) {
        int lo = 0, hi = plan.nbox - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (plan.boxes[mid].start <= (long long)blk) lo = mid; else hi = mid - 1;
        }
        b = lo;
    }
    const TileBox& tb = plan.boxes[b];
    const long long loc = (long long)blk - tb.start;
    const long long ntile = (long long)tb.nt[0] * tb.nt[1];
    long long tile;
    int sg, nsg;
    if (loc < (long long)tb.s * ntile) {
        sg = (int)(loc / ntile);
        tile = loc - (long long)sg * ntile;
        nsg = tile < tb.k1 ? tb.s + 1 : tb.s;
    } else {
        sg = tb.s;
        tile = loc - (long long)tb.s * ntile;
        nsg = tb.s + 1;
    }
    const int tX = (int)(tile % tb.nt[0]), tY = (int)(tile / tb.nt[0]);
    const BoxDesc& B = boxes[b];
    unsigned t = threadIdx.x;
    const int i0 = tb.x0 + tX * (TX - 2), j0 = tb.y0 + tY * (TY - 2);
    const long long L = tb.zhi - tb.zlo + 1;
    const int ks = tb.zlo + (int)(sg * L / nsg), ke = tb.zlo + (int)((sg + 1) * L / nsg);
    const int nb = B.nb, n0 = B.n[0], n1 = B.n[1], n2 = B.n[2];
    const long long sx = 1, sy = B.P[0], sz = (long long)B.P[0] * B.P[1];
    auto inr = [](int v, int lo, int hi) { return v >= lo && v <= hi; };
    // the per-lane conditions as bits of one vector register (see k_vl_stage)
    enum { LB_FX, LB_FY, LB_FZ, LB_C, LB_U, LB_CCB, LB_INT };
    const int sh = a.ccb_lo_shift;
    unsigned lane_bits = 0;
    {
        const int tx = (int)(t % TX), ty = (int)(t / TX), i = i0 + tx, j = j0 + ty;
        // column TX-1's x-faces and row TY-1's y-faces are formed by the next tile
        const bool fx = tx < TX - 1 && inr(i, a.fn_lo, n0 + a.fn_hi) && inr(j, a.ft_lo, n1 + a.ft_hi);
        const bool fy = ty < TY - 1 && inr(j, a.fn_lo, n1 + a.fn_hi) && inr(i, a.ft_lo, n0 + a.ft_hi);
        const bool fz = inr(i, a.ft_lo, n0 + a.ft_hi) && inr(j, a.ft_lo, n1 + a.ft_hi);
        const bool co = tx < TX - 1 && ty < TY - 1 && inr(i, a.c_lo, n0 + a.c_hi) && inr(j, a.c_lo, n1 + a.c_hi);
        const bool up = tx >= 1 && tx < TX - 1 && ty >= 1 && ty < TY - 1 && inr(i, a.u_lo, n0 + a.u_hi) &&
                        inr(j, a.u_lo, n1 + a.u_hi);
        const bool ccb = i >= a.u_lo + sh && j >= a.u_lo + sh;
        const bool in = i >= 1 && j >= 1 && i <= n0 && j <= n1;
        lane_bits = (unsigned)fx << LB_FX | (unsigned)fy << LB_FY | (unsigned)fz << LB_FZ | (unsigned)co << LB_C |
                    (unsigned)up << LB_U | (unsigned)ccb << LB_CCB | (unsigned)in << LB_INT;
    }
    auto lb = [&](int bit) -> bool { return (lane_bits >> bit) & 1u; };
    const double dtdx = a.factor * a.dt[b] / B.dx, cs = a.cs, beta = a.mc_beta;

    auto cell_ok = [&](int ii, int jj, int p) {
        return inr(ii, 1 - nb, n0 + nb) && inr(jj, 1 - nb, n1 + nb) && inr(p, 1 - nb, n2 + nb);
    };
    auto load_cons = [&](int ii, int jj, int p, double* u) {   // zero outside the padded box
        if (cell_ok(ii, jj, p)) {
            const long long c = cell_index(B, ii, jj, p);
#pragma unroll
            for (int f = 0; f < 7; f++) u[f] = a.qf[f][c];
        } else {
#pragma unroll
            for (int f = 0; f < 7; f++) u[f] = 0.0;
        }
    };
    auto to_prims = [&](double* u) {
        const double ir = u[0] != 0.0 ? 1.0 / u[0] : 0.0;
        u[1] = u[1] * ir;
        u[2] = u[2] * ir;
        u[3] = u[3] * ir;
    };
    auto face_b = [&](int d, int ii, int jj, int p) -> double {
        if (!cell_ok(ii, jj, p)) return 0.0;
        return a.bf[d][cell_index(B, ii, jj, p)];
    };
    // the ring cell of slot s (0 .. NR-1): y rows first (coalesced), then x columns
    auto ring_xy = [&](int s, int& rx, int& ry) {
        if (s < 2 * TX) {
            rx = s % TX;
            ry = s < TX ? -1 : TY;
        } else {
            ry = (s - 2 * TX) >> 1;
            rx = (s & 1) ? TX : -1;
        }
    };
    double sm = 0.0, cfl = 0.0;
    double fz[4], dxy[4], dxn[4];   // z flux of the face below; x/y flux differences of the next plane
    double eyx_lo = 0.0, exy_lo = 0.0;   // x face's Ey slot and y face's Ex slot of plane k
    double yez_lo = 0.0;                 // y face E(2,1) of plane k
    double cey_lo = 0.0, vx_lo = 0.0, vz_lo = 0.0;   // centre Ey, m_x/rho, m_z/rho of plane k
    double cey_hi = 0.0, vx_hi = 0.0, vz_hi = 0.0;   // and of plane k+1
    double cex = 0.0, cez = 0.0, cvy = 0.0;          // plane k+1's, on their way to LDS
    double ey_m = 0.0;   // corner Ey of index k-1
    double bz_m = 0.0;
    bool have_bzm = false;
    // z march.  Predictor: plane k's conserved values.  Corrector: plane k's primitives and
    // its limited upper state
    double w0z[6], uLz[6];
#pragma unroll
    for (int f = 0; f < 4; f++) fz[f] = dxy[f] = dxn[f] = 0.0;
#pragma unroll
    for (int r = 0; r < 6; r++) w0z[r] = uLz[r] = 0.0;
    double wbx, wby, wbz;   // face fields of this pass's faces, loaded one pass ahead
    // ring cell loads of slot s for plane p (corrector)
    auto load_ring = [&](int p, unsigned s, double* g) {
        if (!PRED && s < NR) {
            int rx, ry;
            ring_xy((int)s, rx, ry);
            load_cons(i0 + rx, j0 + ry, p, g);
        }
    };
    // a plane's own cell u (ir = 1/rho) and ring cell g into LDS, its centre EMFs and
    // velocities (k_corner's) into registers
    auto fill = [&](const double* u, double ir, double* g, unsigned own, unsigned s) {
        const double r = u[0], m1 = u[1], m2 = u[2], m3 = u[3], b4 = u[4], b5 = u[5], b6 = u[6];
        cex = (b5 * m3 - b6 * m2) * ir;
        cey_hi = (b6 * m1 - b4 * m3) * ir;
        cez = (b4 * m2 - b5 * m1) * ir;
        vx_hi = m1 / r;
        cvy = m2 / r;
        vz_hi = m3 / r;
        if constexpr (PRED) {
            sV[0][own] = vx_hi;
            sV[1][own] = cvy;
            sV[2][own] = vz_hi;
        }
#pragma unroll
        for (int f = 0; f < 7; f++) sW[f][own] = !PRED && f >= 1 && f <= 3 ? u[f] * ir : u[f];
        if (!PRED && s < NR) {
            int rx, ry;
            ring_xy((int)s, rx, ry);
            to_prims(g);
#pragma unroll
            for (int f = 0; f < 7; f++) sW[f][(ry + 1) * PX + rx + 1] = g[f];
        }
    };
    auto recip = [](double r) { return r != 0.0 ? 1.0 / r : 0.0; };
    {
        const int tx = (int)(t % TX), ty = (int)(t / TX), i = i0 + tx, j = j0 + ty;
        double u[7], g[7];
        if (!PRED) {
            load_cons(i, j, ks - 2, u);
            to_prims(u);
#pragma unroll
            for (int r = 0; r < 6; r++) w0z[r] = u[rslot<2>(r)];
        }
        load_cons(i, j, ks - 1, u);
        load_ring(ks - 1, t, g);
        fill(u, recip(u[0]), g, (ty + RING) * PX + tx + RING, t);
        wbx = face_b(0, i, j, ks - 1);
        wby = face_b(1, i, j, ks - 1);
        wbz = face_b(2, i, j, ks - 2);
    }
    __syncthreads();
    // The first pass (k = ks - 2) only forms plane ks - 1, by the same code as every plane.
#pragma unroll 1
    for (int k = ks - 2; k < ke; k++) {
        asm volatile("" : "+v"(lane_bits), "+v"(t));
        const int tx = (int)(t % TX), ty = (int)(t / TX);
        const int i = i0 + tx, j = j0 + ty, own = (ty + RING) * PX + tx + RING;
        const bool live = k >= ks - 1;   // uniform over the workgroup
        const int p = k + 1, q0 = k & 1, q1 = p & 1;
        const bool pt = inr(p, a.ft_lo, n2 + a.ft_hi);
        // ---- A
        // everything of plane k+2, in flight while the faces are solved
        double u[7], g[7];
        const unsigned rs = (t + 64u * (unsigned)k) & (N - 1);   // the ring's wave changes from plane to plane
        load_cons(i, j, k + 2, u);
        load_ring(k + 2, rs, g);
        const double wbx_n = face_b(0, i, j, k + 2), wby_n = face_b(1, i, j, k + 2), wbz_n = face_b(2, i, j, p);
        sC[q1][0][t] = cex;
        sC[q1][1][t] = cez;
        sC[q1][2][t] = cvy;
        double exy_hi = 0.0, eyx_hi = 0.0, yez_hi = 0.0, z0 = 0.0;
        __builtin_amdgcn_sched_barrier(0);
        {   // y-face j+1/2
            double sl[6], sr[6];
            const int up = ty < TY - 1 ? PX : 0, up2 = PRED ? 0 : (ty < TY - 1 ? 2 * PX : PX);
#pragma unroll
            for (int r = 0; r < 6; r++) {
                const int f = rslot<1>(r);
                const double w = sW[f][own], wp = sW[f][own + up];
                if (PRED) {
                    sl[r] = w;
                    sr[r] = wp;
                } else {
                    sl[r] = w + 0.5 * mc_slope(sW[f][own - PX], w, wp, beta);
                    sr[r] = wp - 0.5 * mc_slope(w, wp, sW[f][own + up2], beta);
                }
            }
            if (lb(LB_FY) && pt) {
                double F[7];
                double vl[3], vr[3];
                if constexpr (PRED) {
#pragma unroll
                    for (int r = 0; r < 3; r++) {
                        vl[r] = sV[rslot<1>(r + 1) - 1][t];
                        vr[r] = sV[rslot<1>(r + 1) - 1][t + up];
                    }
                }
                sm = fmax(sm, near_solve<RS, PRED>(sl, sr, vl, vr, wby, cs, F));
                sF[0][t] = F[0]; sF[2][t] = F[1]; sF[3][t] = F[2]; sF[1][t] = F[3];
                exy_hi = -F[5];
                yez_hi = F[6];
            } else {
                sF[0][t] = sF[1][t] = sF[2][t] = sF[3][t] = 0.0;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        {   // x-face i+1/2: the upper neighbour's (lower limited) state from lane + 1
            double sl[6], sr[6], fx[4];
#pragma unroll
            for (int r = 0; r < 6; r++) {
                const int f = rslot<0>(r);
                const double w = sW[f][own];
                if (PRED) {
                    sl[r] = w;
                    sr[r] = lane_next_d(w);
                } else {
                    const double d = mc_slope(sW[f][own - 1], w, sW[f][own + 1], beta);
                    sl[r] = w + 0.5 * d;
                    sr[r] = lane_next_d(w - 0.5 * d);
                }
            }
            double xez = 0.0, vl[3], vr[3];
            if constexpr (PRED) {
                vl[0] = vx_hi;
                vl[1] = sV[1][t];
                vl[2] = vz_hi;
#pragma unroll
                for (int r = 0; r < 3; r++) vr[r] = lane_next_d(vl[r]);
            }
            if (lb(LB_FX) && pt) {
                double F[7];
                sm = fmax(sm, near_solve<RS, PRED>(sl, sr, vl, vr, wbx, cs, F));
                fx[0] = F[0]; fx[1] = F[1]; fx[2] = F[2]; fx[3] = F[3];
                xez = -F[5];
                eyx_hi = F[6];
            } else {
                fx[0] = fx[1] = fx[2] = fx[3] = 0.0;
            }
            sEf[q1][t] = xez;
#pragma unroll
            for (int f = 0; f < 4; f++) dxn[f] = fx[f] - lane_prev_d(fx[f]);
        }
        __builtin_amdgcn_sched_barrier(0);
        double ir = 0.0;
        {   // z-face k+1/2
            double sl[6], sr[6];
            if (PRED) {
#pragma unroll
                for (int r = 0; r < 6; r++) {
                    sl[r] = w0z[r];
                    sr[r] = w0z[r] = sW[rslot<2>(r)][own];
                }
            } else {
                ir = recip(u[0]);
                const double P[7] = {u[0], u[1] * ir, u[2] * ir, u[3] * ir, u[4], u[5], u[6]};
#pragma unroll
                for (int r = 0; r < 6; r++) {
                    const double w = sW[rslot<2>(r)][own];
                    const double d = mc_slope(w0z[r], w, P[rslot<2>(r)], beta);
                    sl[r] = uLz[r];
                    sr[r] = w - 0.5 * d;
                    uLz[r] = w + 0.5 * d;
                    w0z[r] = w;
                }
            }
            double fu[4] = {0.0, 0.0, 0.0, 0.0}, z1 = 0.0;
            if (live && lb(LB_FZ) && inr(k, a.fn_lo, n2 + a.fn_hi)) {
                double F[7];
                const double vl[3] = {vz_lo, vx_lo, sC[q0][2][t]}, vr[3] = {vz_hi, vx_hi, sC[q1][2][t]};
                sm = fmax(sm, near_solve<RS, PRED>(sl, sr, vl, vr, wbz, cs, F));
                fu[0] = F[0]; fu[3] = F[1]; fu[1] = F[2]; fu[2] = F[3];
                z0 = -F[5];
                z1 = F[6];
            }
            sEz3[t] = z1;
#pragma unroll
            for (int f = 0; f < 4; f++) {   // the flux divergence of plane k
                dxy[f] = dxy[f] + (fu[f] - fz[f]);
                fz[f] = fu[f];
            }
        }
        __syncthreads();
        // ---- D: the update's inputs first, then the corner EMFs of index k, the flux
        // differences of plane k+1, and plane k+2 into LDS
        double div[4];
#pragma unroll
        for (int f = 0; f < 4; f++) div[f] = dxy[f];
        const bool upd = k >= ks && lb(LB_U) && inr(k, a.u_lo, n2 + a.u_hi);
        const bool ccb = lb(LB_CCB) && k >= a.u_lo + sh;
        double pq[4] = {0.0, 0.0, 0.0, 0.0};
        double pb[3] = {0.0, 0.0, 0.0}, pbm[3] = {0.0, 0.0, 0.0};
        if (upd) {
            const long long c = cell_index(B, i, j, k);
#pragma unroll
            for (int f = 0; f < 4; f++) pq[f] = PRED ? a.qf[f][c] : a.src.q[f][c];   // predictor: the flux state is the base
#pragma unroll
            for (int d = 0; d < 3; d++) pb[d] = a.src.b[d][c];
            if (ccb) {
                pbm[0] = a.src.b[0][c - sx];
                pbm[1] = a.src.b[1][c - sy];
                if (!have_bzm) pbm[2] = a.src.b[2][c - sz];
            }
        }
        double ey = 0.0;   // corner Ey of index k
        {
            // x-neighbours' values (lane shifts, all lanes take part)
            const double vx_n = lane_next_d(vx_lo), yez_n = lane_next_d(yez_lo), z0_n = lane_next_d(z0),
                         cl_n = lane_next_d(cey_lo), ch_n = lane_next_d(cey_hi);
            if (live && lb(LB_C) && inr(k, a.c_lo, n2 + a.c_hi)) {
                const double vx = 0.5 * (vx_lo + vx_n), vy = 0.5 * (sC[q0][2][t] + sC[q0][2][t + TX]);
                const double vz = 0.5 * (vz_lo + vz_hi);
                double a14, a34, b14, b34;
                {   // Ez at (i+1/2, j+1/2, k); the factor 2 of k_corner's differences taken out
                    const double e00 = sC[q0][1][t], e10 = sC[q0][1][t + 1], e01 = sC[q0][1][t + TX],
                                 e11 = sC[q0][1][t + TX + 1];
                    const double y0 = yez_lo, y1 = yez_n, x0 = sEf[q0][t], x1 = sEf[q0][t + TX];
                    upw(vx, y0 - e00, y1 - e10, e01 - y0, e11 - y1, a14, a34);
                    upw(vy, x0 - e00, x1 - e01, e10 - x0, e11 - x1, b14, b34);
                    sEz[t] = (0.25 * (x0 + x1 + y0 + y1) + 0.25 * ((a14 - a34) + (b14 - b34)));
                }
                {   // Ey at (i+1/2, j, k+1/2)
                    const double x0 = eyx_lo, x1 = eyx_hi;
                    upw(vx, z0 - cey_lo, z0_n - cl_n, cey_hi - z0, ch_n - z0_n, a14, a34);
                    upw(vz, x0 - cey_lo, x1 - cey_hi, cl_n - x0, ch_n - x1, b14, b34);
                    ey = (0.25 * (x0 + x1 + z0 + z0_n) + 0.25 * ((a14 - a34) + (b14 - b34)));
                }
                {   // Ex at (i, j+1/2, k+1/2)
                    const double e00 = sC[q0][0][t], e10 = sC[q0][0][t + TX], e01 = sC[q1][0][t], e11 = sC[q1][0][t + TX];
                    const double w0 = sEz3[t], w1 = sEz3[t + TX], y0 = exy_lo, y1 = exy_hi;
                    upw(vy, w0 - e00, w1 - e10, e01 - w0, e11 - w1, a14, a34);
                    upw(vz, y0 - e00, y1 - e01, e10 - y0, e11 - y1, b14, b34);
                    sEx[q0][t] = (0.25 * (y0 + y1 + w0 + w1) + 0.25 * ((a14 - a34) + (b14 - b34)));
                }
            }
        }
        if (lb(LB_U)) {
#pragma unroll
            for (int f = 0; f < 4; f++) dxy[f] = dxn[f] + (sF[f][t] - sF[f][t - TX]);
        }
        cey_lo = cey_hi;
        vx_lo = vx_hi;
        vz_lo = vz_hi;
        eyx_lo = eyx_hi;
        exy_lo = exy_hi;
        yez_lo = yez_hi;
        wbx = wbx_n;
        wby = wby_n;
        wbz = wbz_n;
        if (PRED) ir = recip(u[0]);
        fill(u, ir, g, own, rs);
        __syncthreads();
        // ---- G: update of plane k (k_update_z's arithmetic)
        const double ey_x = lane_prev_d(ey), eyx_m = lane_prev_d(ey_m);
        if (upd) {
            const long long c = cell_index(B, i, j, k);
            double nq[7], oq[4];
#pragma unroll
            for (int f = 0; f < 4; f++) {
                const double q0v = pq[f];
                oq[f] = q0v;
                double v = q0v - dtdx * div[f];
                if (f == 0 && v < MIN_DENS) {
                    v = MIN_DENS;
                    atomicAdd(a.floor_count, a.img ? floor_images(n0, n1, n2, i, j, k, a.img_lo, a.img_hi) : 1u);
                }
                a.dst.q[f][c] = v;
                nq[f] = v;
            }
            const double ex = sEx[q0][t], ex_y = sEx[q0][t - TX], ez = sEz[t], ez_y = sEz[t - TX], ez_x = sEz[t - 1];
            const double ex_m = sEx[q1][t], exy_m = sEx[q1][t - TX];
            const double bx = pb[0] - dtdx * ((ez - ez_y) - (ey - ey_m));
            const double by = pb[1] - dtdx * ((ex - ex_m) - (ez - ez_x));
            const double bz = pb[2] - dtdx * ((ey - ey_x) - (ex - ex_y));
            a.dst.b[0][c] = bx;
            a.dst.b[1][c] = by;
            a.dst.b[2][c] = bz;
            if (ccb) {
                const double ez_xy = sEz[t - 1 - TX];
                const double bxm = pbm[0] - dtdx * ((ez_x - ez_xy) - (ey_x - eyx_m));
                const double bym = pbm[1] - dtdx * ((ex_y - exy_m) - (ez_y - ez_xy));
                if (!have_bzm) bz_m = pbm[2] - dtdx * ((ey_m - eyx_m) - (ex_m - exy_m));
                nq[4] = (0.5 * (bx + bxm));
                nq[5] = (0.5 * (by + bym));
                nq[6] = (0.5 * (bz + bz_m));
            } else {
#pragma unroll
                for (int f = 4; f < 7; f++) nq[f] = PRED ? a.qf[f][c] : a.src.q[f][c];
            }
#pragma unroll
            for (int f = 4; f < 7; f++) a.dst.q[f][c] = nq[f];
            bz_m = bz;
            have_bzm = true;
            if (a.pvel[0] != nullptr) {   // passive velocities (copy_velocity's arithmetic)
                const double io = 1.0 / oq[0];
                if (PRED) {
#pragma unroll
                    for (int d = 0; d < 3; d++) a.pvel[d][c] = oq[1 + d] * io;
                } else {
                    const double in = 1.0 / nq[0];
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        const double vo = oq[1 + d] * io;
                        a.pvel[d][c] = 0.5 * (vo + nq[1 + d] * in);
                    }
                }
            }
            if (!PRED && a.cmax != nullptr && lb(LB_INT) && k >= 1 && k <= n2) cfl = fmax(cfl, cell_fast_speed(nq, a.cs));
        } else {
            have_bzm = false;
        }
        ey_m = ey;
    }
    atomic_max_nonneg(a.smax, b, sm);
    if (!PRED && a.cmax != nullptr) atomic_max_nonneg(a.cmax, b, cfl);
}

template <int RS, bool PRED, class F>
auto vl_near_shape(int shape, F f) {
    if (shape == 0) return f(k_vl_near<RS, PRED, vs_tx(0), vs_ty(0)>, vs_tx(0) * vs_ty(0));
    return f(k_vl_near<RS, PRED, vs_tx(1), vs_ty(1)>, vs_tx(1) * vs_ty(1));
}
template <int RS, bool PRED>
void launch_vl_near(hipStream_t st, const BoxDesc* boxes, const TilePlan& plan, const StageArgs<double>& a, int shape) {
    if (plan.total <= 0) return;
    vl_near_shape<RS, PRED>(shape, [&](auto kern, int n) {
        hipLaunchKernelGGL(kern, dim3((unsigned)plan.total), dim3(n), 0, st, boxes, plan, a);
    });
}
template <int RS, bool PRED>
int vl_near_blocks_per_cu(int shape) {
    return vl_near_shape<RS, PRED>(shape, [&](auto kern, int nt) {
        int n = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, nt, 0);
        return e == hipSuccess && n > 0 ? n : 1;
    });
}

#define IMHD_INST_NEAR(RS, PRED)                                                                                           \
    template void launch_vl_near<RS, PRED>(hipStream_t, const BoxDesc*, const TilePlan&, const StageArgs<double>&, int); \
    template int vl_near_blocks_per_cu<RS, PRED>(int);

}  // namespace imhd
