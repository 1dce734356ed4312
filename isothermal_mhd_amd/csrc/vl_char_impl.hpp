// Fused corrector of the VL integrator with characteristic PPM (the reference's default
// reconstruction, vanleer_mod.f90:941-1141, 1595-1818): one launch does the directional
// fluxes, the upwind corner EMFs (:1884-2076) and the conservative + CT update (:2080-2259),
// as k_vl_stage does for the other stages, with the same tiles, z-segments, masks and
// per-value arithmetic.
//
// What bounds it is the reconstruction's arithmetic.  The edge value of cell c towards its
// upper face,
//     E(c) = (W_c + W_{c+1}) / 2 - delw_c / 6,
// needs the 6 x 6 eigenvectors of cell c and its projections of cells c-1 .. c+2, and a face
// c+1/2 needs E(c-1), E(c), E(c+1).  Formed per face that is nine edge values per cell and
// plane; here each cell forms its own three (one per direction) and the faces share them:
//   x  the lower neighbour's E and the upper neighbour's limited state by lane shift;
//   y  E through LDS;
//   z  E and the limited upper state carried from plane to plane of the march.
// The cells just below a tile (column -1, row -1) belong to no thread: one wave, another
// each plane, forms their E, so the tiles keep the two-column overlap of the other stages.
//
// Per plane k of the march (the primitives of plane k+1, with two ring cells on every side,
// are in LDS):
//   A1  E of plane k+1 along y and z; z-face k+1/2; centre EMFs of plane k+1
//   A2  y-faces, then E along x and the x-faces, of plane k+1
//   D   corner EMFs of index k; the primitives of plane k+2 replace plane k+1's
//   G   update of plane k
// with a barrier after A1, A2 and D.  Scheduling fences keep the phases' working sets apart,
// and the thread index is marked as rewritten each plane, so that LDS and global addresses
// are formed where they are used: hoisted out of the march they took 70 registers.  FP64 reads
// the own column's planes k, k+2 and k+3 again from L2 each plane for the same reason; FP32 has
// the registers to carry them and loads plane k+3 only, at the start of the pass.
// FP64: two workgroups per CU (75 KB of LDS per 16 x 16 tile, 256 registers): the 63 registers
// that spill cost less than the second workgroup gains (128^3, full ranges in four rounds of
// segments: 1.10 ms per launch, against 1.36 ms with one workgroup and nothing spilled).
//
// Measured per launch at 128^3 (HLLD), against the per-face form: 2.02 -> 1.10 ms, 0.95 over the
// ranges of a native step in one round of segments; the VALU is busy in 57 % of the cycles.
//
// FP32 is the same kernel with the fused operations of the per-face form written out
// (char_edge, ppm_edge, char_solve), so that its results keep their bits: a rounding moved in
// an edge value turns up as a different limiter branch in single cells.  Per launch at 256^3
// (HLLD) 4.02 -> 2.76 ms with 16 x 16 tiles, 2.60 with the own column carried.  It is bound by
// VALU issue (5206 instructions per cell, the VALU busy in 90 % of the cycles);
// four waves per SIMD, by lane shifts in place of 8 KB of LDS, spill 99 registers: 3.5 ms.
#pragma once
#include "vl_stage_impl.hpp"

namespace imhd {

// E(c) from W[0..3] = cells c-1 .. c+2 and the cell's upper face field: the values of
// prim_eigvecs and char_delw bit for bit, formed a wave pair at a time so that few are live.
// The two waves of a pair have eigenvectors that differ in signs only; a product's sign is
// exact, so they share their products and differ in the signs of the additions.  The zero
// entries of the Alfven pair stay as products with zero (they carry a NaN or an infinity).
__device__ __forceinline__ void char_edge(const double (*W)[6], double wb, double cs, double beta, double* E) {
    const double asqr = cs * cs;
    const double rho = W[1][0], irho = 1.0 / rho, rhos = sqrt(rho), irhos = 1.0 / rhos;
    const double bx = irhos * wb, by = irhos * W[1][4], bz = irhos * W[1][5];
    const double bsqr = bx * bx + by * by + bz * bz;
    const double btsqr = by * by + bz * bz;
    const double tmp1 = asqr + bsqr, x = asqr - bsqr;
    const double tmp2 = sqrt(x * x + 4.0 * asqr * btsqr);
    const double cslow = sqrt(max2(0.0, 0.5 * (tmp1 - tmp2)));
    const double cf = sqrt(0.5 * (tmp1 + tmp2));
    double af, as;
    if (fabs(cf * cf - cslow * cslow) < ZERO) { af = 1.0; as = 0.0; }
    else {
        af = sqrt(max2((asqr - cslow * cslow) / (cf * cf - cslow * cslow), 0.0));
        as = sqrt(max2((cf * cf - asqr) / (cf * cf - cslow * cslow), 0.0));
    }
    double n1, n2;
    if (btsqr < ZERO) { n1 = 1.0 / sqrt(2.0); n2 = n1; }
    else { n1 = by / sqrt(btsqr); n2 = bz / sqrt(btsqr); }
    const double S = sgn1(bx);
    const double Cff = cf * af, Css = cslow * as, Qf = cf * af * S, Qs = cslow * as * S;
    const double Af = cs * af * rhos, As = cs * as * rhos;
    const double Nf = 0.5 / asqr;
    double dm[6];
    auto slope = [&](double aL1, double aC, double aR1, double aR2) {
        const double dL1 = aC - aL1, dR1 = aR1 - aC, dC1 = 0.5 * (dL1 + dR1);
        const double dR2 = aR2 - aR1, dC2 = 0.5 * (dR1 + dR2);
        // mc_lim without its branch (sign(dC) m, m >= 0, is copysign(m, dC) exactly)
        const double m1 = copysign(min3(beta * fabs(dL1), beta * fabs(dR1), fabs(dC1)), dC1);
        const double m2 = copysign(min3(beta * fabs(dR1), beta * fabs(dR2), fabs(dC2)), dC2);
        return (dR1 * dR2 > 0.0 ? m2 : 0.0) - (dL1 * dR1 > 0.0 ? m1 : 0.0);
    };
    double lo[4], hi[4];
    __builtin_amdgcn_sched_barrier(0);
    {   // fast: L0 = (a, -b, c, d, e, f), L5 = (a, b, -c, -d, e, f)
        const double l0 = Nf * af * asqr * irho, l1 = Nf * Cff, l2 = Nf * Qs * n1, l3 = Nf * Qs * n2,
                     l4 = Nf * As * n1 * irho, l5 = Nf * As * n2 * irho;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const double p0 = l0 * W[m][0], p1 = l1 * W[m][1], p2 = l2 * W[m][2], p3 = l3 * W[m][3], p4 = l4 * W[m][4],
                         p5 = l5 * W[m][5];
            lo[m] = p0 - p1 + p2 + p3 + p4 + p5;
            hi[m] = p0 + p1 - p2 - p3 + p4 + p5;
        }
        dm[0] = slope(lo[0], lo[1], lo[2], lo[3]);
        dm[5] = slope(hi[0], hi[1], hi[2], hi[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
    {   // slow: L2 = (a, -b, -c, -d, -e, -f), L3 = (a, b, c, d, -e, -f)
        const double l0 = Nf * as * asqr * irho, l1 = Nf * Css, l2 = Nf * Qf * n1, l3 = Nf * Qf * n2,
                     l4 = Nf * Af * n1 * irho, l5 = Nf * Af * n2 * irho;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const double p0 = l0 * W[m][0], p1 = l1 * W[m][1], p2 = l2 * W[m][2], p3 = l3 * W[m][3], p4 = l4 * W[m][4],
                         p5 = l5 * W[m][5];
            lo[m] = p0 - p1 - p2 - p3 - p4 - p5;
            hi[m] = p0 + p1 + p2 + p3 - p4 - p5;
        }
        dm[2] = slope(lo[0], lo[1], lo[2], lo[3]);
        dm[3] = slope(hi[0], hi[1], hi[2], hi[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
    {   // Alfven: L1 = (0, 0, -c, d, -e, f), L4 = (0, 0, c, -d, -e, f)
        const double l2 = 0.5 * n2, l3 = 0.5 * n1, l4 = 0.5 * n2 * S * irhos, l5 = 0.5 * n1 * S * irhos;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const double z = 0.0 * W[m][0] + 0.0 * W[m][1], p2 = l2 * W[m][2], p3 = l3 * W[m][3], p4 = l4 * W[m][4],
                         p5 = l5 * W[m][5];
            lo[m] = z - p2 + p3 - p4 + p5;
            hi[m] = z + p2 - p3 - p4 + p5;
        }
        dm[1] = slope(lo[0], lo[1], lo[2], lo[3]);
        dm[4] = slope(hi[0], hi[1], hi[2], hi[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
    const double r2 = n2 * S * rhos, r3 = n1 * S * rhos;   // Alfven field entries
    double d[6];
    d[0] = dm[0] * (rho * af) + dm[1] * 0.0 + dm[2] * (rho * as) + dm[3] * (rho * as) + dm[4] * 0.0 + dm[5] * (rho * af);
    d[1] = dm[0] * -Cff + dm[1] * 0.0 + dm[2] * -Css + dm[3] * Css + dm[4] * 0.0 + dm[5] * Cff;
    d[2] = dm[0] * (Qs * n1) + dm[1] * -n2 + dm[2] * (-Qf * n1) + dm[3] * (Qf * n1) + dm[4] * n2 + dm[5] * (-Qs * n1);
    d[3] = dm[0] * (Qs * n2) + dm[1] * n1 + dm[2] * (-Qf * n2) + dm[3] * (Qf * n2) + dm[4] * -n1 + dm[5] * (-Qs * n2);
    d[4] = dm[0] * (As * n1) + dm[1] * -r2 + dm[2] * (-Af * n1) + dm[3] * (-Af * n1) + dm[4] * -r2 + dm[5] * (As * n1);
    d[5] = dm[0] * (As * n2) + dm[1] * r3 + dm[2] * (-Af * n2) + dm[3] * (-Af * n2) + dm[4] * r3 + dm[5] * (As * n2);
    const double sixth = 1.0 / 6.0;
#pragma unroll
    for (int m = 0; m < 6; m++) E[m] = 0.5 * (W[1][m] + W[2][m]) - sixth * d[m];
}
// The FP32 edge value, with the roundings that the per-face form (char_delw and ppm_states,
// compiled with FMA contraction) has: contraction is off here and the fused operations are
// written out, so that the cell's one value is the one that each of its faces formed there.
// A wave pair's first projection was fused, its second added the rounded products.
__device__ __forceinline__ void char_edge(const float (*W)[6], float wb, float cs, float beta, float* E) {
#pragma clang fp contract(off)
    const float asqr = cs * cs;
    const float rho = W[1][0], irho = __builtin_amdgcn_rcpf(rho), rhos = fsqrt(rho), irhos = __builtin_amdgcn_rcpf(rhos);
    const float bx = irhos * wb, by = irhos * W[1][4], bz = irhos * W[1][5];
    const float bsqr = fmaf(bz, bz, fmaf(by, by, bx * bx));
    const float btsqr = fmaf(by, by, bz * bz);
    const float tmp1 = asqr + bsqr, x = asqr - bsqr;
    const float tmp2 = fsqrt(fmaf(4.0f * asqr, btsqr, x * x));
    const float cslow = fsqrt(max2(0.0f, 0.5f * (tmp1 - tmp2)));
    const float cf = fsqrt(0.5f * (tmp1 + tmp2));
    const float cs2 = cslow * cslow, cf2 = cf * cf, dif = fmaf(cf, cf, -cs2), idif = __builtin_amdgcn_rcpf(dif);
    const bool same = fabs(dif) < (float)ZERO;
    const float af = same ? 1.0f : fsqrt(max2((asqr - cs2) * idif, 0.0f));
    const float as = same ? 0.0f : fsqrt(max2((cf2 - asqr) * idif, 0.0f));
    const bool flat = btsqr < (float)ZERO;
    const float ibt = __builtin_amdgcn_rsqf(flat ? 2.0f : btsqr);
    const float n1 = flat ? ibt : by * ibt, n2 = flat ? ibt : bz * ibt;
    const float S = sgn1(bx);
    const float Cff = cf * af, Css = cslow * as, Qf = Cff * S, Qs = Css * S;
    const float Af = cs * af * rhos, As = cs * as * rhos;
    const float Nf = 0.5f * __builtin_amdgcn_rcpf(asqr);
    float dm[6], lo[4], hi[4];
    auto slope = [&](const float* v) {
        const float dL1 = v[1] - v[0], dR1 = v[2] - v[1], dC1 = 0.5f * (dL1 + dR1);
        const float dR2 = v[3] - v[2], dC2 = 0.5f * (dR1 + dR2);
        // mc_lim without its branch (sign(dC) m, m >= 0, is copysign(m, dC) exactly)
        const float m1 = copysign(min3(beta * fabs(dL1), beta * fabs(dR1), fabs(dC1)), dC1);
        const float m2 = copysign(min3(beta * fabs(dR1), beta * fabs(dR2), fabs(dC2)), dC2);
        return (dR1 * dR2 > 0.0f ? m2 : 0.0f) - (dL1 * dR1 > 0.0f ? m1 : 0.0f);
    };
    {   // fast: L0 = (a, -b, c, d, e, f), L5 = (a, b, -c, -d, e, f)
        const float l0 = Nf * af * asqr * irho, l1 = Nf * Cff, l2 = Nf * Qs * n1, l3 = Nf * Qs * n2,
                    l4 = Nf * As * n1 * irho, l5 = Nf * As * n2 * irho;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const float* w = W[m];
            const float p1 = w[1] * l1;
            lo[m] = fmaf(w[5], l5, fmaf(w[4], l4, fmaf(w[3], l3, fmaf(w[2], l2, fmaf(w[0], l0, -p1)))));
            hi[m] = w[0] * l0 + p1 - w[2] * l2 - w[3] * l3 + w[4] * l4 + w[5] * l5;
        }
        dm[0] = slope(lo);
        dm[5] = slope(hi);
    }
    __builtin_amdgcn_sched_barrier(0);
    {   // slow: L2 = (a, -b, -c, -d, -e, -f), L3 = (a, b, c, d, -e, -f)
        const float l0 = Nf * as * asqr * irho, l1 = Nf * Css, l2 = Nf * Qf * n1, l3 = Nf * Qf * n2,
                    l4 = Nf * Af * n1 * irho, l5 = Nf * Af * n2 * irho;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const float* w = W[m];
            const float p1 = w[1] * l1;
            lo[m] = fmaf(-w[5], l5, fmaf(-w[4], l4, fmaf(-w[3], l3, fmaf(-w[2], l2, fmaf(w[0], l0, -p1)))));
            hi[m] = w[0] * l0 + p1 + w[2] * l2 + w[3] * l3 - w[4] * l4 - w[5] * l5;
        }
        dm[2] = slope(lo);
        dm[3] = slope(hi);
    }
    __builtin_amdgcn_sched_barrier(0);
    {   // Alfven: L1 = (0, 0, -c, d, -e, f), L4 = (0, 0, c, -d, -e, f)
        const float l2 = 0.5f * n2, l3 = 0.5f * n1, l4 = l2 * S * irhos, l5 = l3 * S * irhos;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const float* w = W[m];
            const float z = fmaf(w[0], 0.0f, w[1] * 0.0f);
            lo[m] = fmaf(w[5], l5, fmaf(-w[4], l4, fmaf(w[3], l3, fmaf(-w[2], l2, z))));
            hi[m] = z + w[2] * l2 - w[3] * l3 - w[4] * l4 + w[5] * l5;
        }
        dm[1] = slope(lo);
        dm[4] = slope(hi);
    }
    __builtin_amdgcn_sched_barrier(0);
    const float r2 = n2 * S * rhos, r3 = n1 * S * rhos;   // Alfven field entries
    float d[6];
    auto comb = [&](float r0, float r1, float r2_, float r3_, float r4, float r5) {
        return fmaf(r5, dm[5], fmaf(r4, dm[4], fmaf(r3_, dm[3], fmaf(r2_, dm[2], fmaf(r0, dm[0], r1 * dm[1])))));
    };
    d[0] = comb(rho * af, 0.0f, rho * as, rho * as, 0.0f, rho * af);
    d[1] = comb(-Cff, 0.0f, -Css, Css, 0.0f, Cff);
    d[2] = comb(Qs * n1, -n2, -(Qf * n1), Qf * n1, n2, -(Qs * n1));
    d[3] = comb(Qs * n2, n1, -(Qf * n2), Qf * n2, -n1, -(Qs * n2));
    d[4] = comb(As * n1, -r2, -(Af * n1), -(Af * n1), -r2, As * n1);
    d[5] = comb(As * n2, r3, -(Af * n2), -(Af * n2), r3, As * n2);
    const float sixth = __builtin_amdgcn_rcpf(6.0f);
#pragma unroll
    for (int m = 0; m < 6; m++) E[m] = fmaf(W[1][m] + W[2][m], 0.5f, -(d[m] * sixth));
}
// Limited edge values of a cell from its raw ones, the lower (UP = false) or the upper
// (vanleer_mod.f90:1724-1743): ppm_monotone's arithmetic without branches (a wavefront's
// lanes rarely agree), in FP32 with the fused operations that its branches had.
template <bool UP>
__device__ __forceinline__ double ppm_edge(double w, double wL, double wR) {
    const double tmp1 = (wR - w) * (w - wL);
    const double tmp2 = 6.0 * (wR - wL) * (w - 0.5 * (wL + wR));
    const double d = wR - wL, tmp3 = d * d;
    const double e = UP ? (tmp2 < -tmp3 ? 3.0 * w - 2.0 * wL : wR) : (tmp2 > tmp3 ? 3.0 * w - 2.0 * wR : wL);
    return tmp1 <= 0.0 ? w : e;
}
template <bool UP>
__device__ __forceinline__ float ppm_edge(float w, float wL, float wR) {
#pragma clang fp contract(off)
    const float tmp1 = (wR - w) * (w - wL);
    const float d = wR - wL, tmp3 = d * d;
    const float tmp2 = 6.0f * d * fmaf(-0.5f, wL + wR, w);
    const float e = UP ? (tmp2 < -tmp3 ? fmaf(3.0f, w, -2.0f * wL) : wR) : (tmp2 > tmp3 ? fmaf(3.0f, w, -2.0f * wR) : wL);
    return tmp1 <= 0.0f ? w : e;
}
// Interface states (six rotated primitives each) to a flux, as the per-face form does it:
// FP32 divides the momenta by rho again, FP64 as plm_solve
template <class real, int RS>
__device__ __forceinline__ real char_solve(const real* sl, const real* sr, real wb, real cs, real* F) {
    if constexpr (sizeof(real) == 8) {
        return plm_solve<real, RS>(sl, sr, wb, cs, F);
    } else {
        const real uL[7] = {sl[0], sl[1] * sl[0], sl[2] * sl[0], sl[3] * sl[0], wb, sl[4], sl[5]};
        const real uR[7] = {sr[0], sr[1] * sr[0], sr[2] * sr[0], sr[3] * sr[0], wb, sr[4], sr[5]};
        real smax = real(0);
        if constexpr (RS == RS_HLLD) hlld<real, false, true>(uL, uR, cs * cs, F, smax);
        else if constexpr (RS == RS_HLLE) hlle<real, false, true>(uL, uR, cs * cs, F, smax);
        else roe<real, true>(uL, uR, cs, F, smax);
        return smax;
    }
}
// cells the ring of a tile holds: columns -2, -1, TX, TX + 1 and rows -2, -1, TY, TY + 1
// (no corners: nothing reads them)
template <int TX, int TY>
constexpr int vc_ring() { return 4 * (TX + TY); }

__device__ __forceinline__ double lane_prev_r(double x) { return lane_prev_d(x); }
__device__ __forceinline__ double lane_next_r(double x) { return lane_next_d(x); }
__device__ __forceinline__ float lane_prev_r(float x) { return lane_prev(x); }
__device__ __forceinline__ float lane_next_r(float x) { return lane_next(x); }

// Waves per SIMD (above).  FP64: two, 75 KB of LDS per 16 x 16 tile and 256 registers.  FP32: 45
// KB per 16 x 16 tile and 168 registers, three; 32 x 16 (88 KB) fits one workgroup, at two.
template <class real, int N>
constexpr int vc_waves() { return sizeof(real) == 4 && N == 256 ? 3 : 2; }

// Difference of two faces' fluxes, each rounded by itself (the other stages' fluxes are, on
// their way through LDS): a flux that ends in a product is not fused into it
template <class real>
__device__ __forceinline__ real face_diff(real hi, real lo) {
#pragma clang fp contract(off)
    return hi - lo;
}

#define VC_WAVES (vc_waves<real, TX * TY>())
template <class real, int RS, int TX, int TY>
__global__ __launch_bounds__(TX * TY, VC_WAVES) void k_vl_char(const BoxDesc* __restrict__ boxes,
                                                                      TilePlan plan, StageArgs<real> a) {
    constexpr int N = TX * TY, NW = N / 64, PX = TX + 4, PY = TY + 4, NR = vc_ring<TX, TY>();
    static_assert(64 % TX == 0 && NR <= N && TX + TY <= 64, "tile shape");
    __shared__ real sW[7][PY * PX];       // primitives of plane k+1 (global order) with the ring
    __shared__ real sEy[6][(TY + 1) * TX];   // E of the y direction, rows -1 .. TY-1 (rotated)
    __shared__ real sEx[6][TY];           // E of the x direction, column -1
    __shared__ real sF[4][N];             // y-face fluxes of plane k+1, global order
    __shared__ real sEf[2][N];            // plane k: x face E(2,0); y face E(2,1)
    __shared__ real sEz3[2][N];           // z face k+1/2: E(1,1), E(0,1)
    __shared__ double sC[2][2][N];        // [plane parity] centre Ex, Ey
    __shared__ double sV[3][N];           // plane k: centre Ez, m_x/rho, m_y/rho
    __shared__ real sEz[N];               // corner Ez of plane k
    __shared__ real sEc[2][2][N];         // [index parity] corner Ex, Ey

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
    enum { LB_CELL, LB_FX, LB_FY, LB_FZ, LB_C, LB_U, LB_CCB, LB_INT, LB_X0 };
    const int sh = a.ccb_lo_shift;
    unsigned lane_bits = 0;
    {
        const int tx = (int)(t % TX), ty = (int)(t / TX), i = i0 + tx, j = j0 + ty;
        const bool cell_ij = inr(i, 1 - nb, n0 + nb) && inr(j, 1 - nb, n1 + nb);
        // column TX-1's x-faces and row TY-1's y-faces are formed by the next tile
        const bool fx = tx < TX - 1 && inr(i, a.fn_lo, n0 + a.fn_hi) && inr(j, a.ft_lo, n1 + a.ft_hi);
        const bool fy = ty < TY - 1 && inr(j, a.fn_lo, n1 + a.fn_hi) && inr(i, a.ft_lo, n0 + a.ft_hi);
        const bool fz = inr(i, a.ft_lo, n0 + a.ft_hi) && inr(j, a.ft_lo, n1 + a.ft_hi);
        const bool co = tx < TX - 1 && ty < TY - 1 && inr(i, a.c_lo, n0 + a.c_hi) && inr(j, a.c_lo, n1 + a.c_hi);
        const bool up = tx >= 1 && tx < TX - 1 && ty >= 1 && ty < TY - 1 && inr(i, a.u_lo, n0 + a.u_hi) &&
                        inr(j, a.u_lo, n1 + a.u_hi);
        const bool ccb = i >= a.u_lo + sh && j >= a.u_lo + sh;
        const bool in = i >= 1 && j >= 1 && i <= n0 && j <= n1;
        lane_bits = (unsigned)cell_ij << LB_CELL | (unsigned)fx << LB_FX | (unsigned)fy << LB_FY | (unsigned)fz << LB_FZ |
                    (unsigned)co << LB_C | (unsigned)up << LB_U | (unsigned)ccb << LB_CCB | (unsigned)in << LB_INT |
                    (unsigned)(tx == 0) << LB_X0;
    }
    auto lb = [&](int bit) -> bool { return (lane_bits >> bit) & 1u; };
    const double dtd = a.factor * a.dt[b] / B.dx;
    const real dtdx = (real)dtd, cs = (real)a.cs, beta = (real)a.mc_beta;

    auto cell_ok = [&](int ii, int jj, int p) {
        return inr(ii, 1 - nb, n0 + nb) && inr(jj, 1 - nb, n1 + nb) && inr(p, 1 - nb, n2 + nb);
    };
    auto load_cons = [&](int ii, int jj, int p, real* u) {   // zero outside the padded box
        if (cell_ok(ii, jj, p)) {
            const long long c = cell_index(B, ii, jj, p);
#pragma unroll
            for (int f = 0; f < 7; f++) u[f] = a.qf[f][c];
        } else {
#pragma unroll
            for (int f = 0; f < 7; f++) u[f] = real(0);
        }
    };
    auto to_prims = [&](real* u) {
        const real ir = u[0] != real(0) ? fdiv(real(1), u[0]) : real(0);
        u[1] = u[1] * ir;
        u[2] = u[2] * ir;
        u[3] = u[3] * ir;
    };
    auto face_b = [&](int d, int ii, int jj, int p) -> real {
        if (!cell_ok(ii, jj, p)) return real(0);
        const long long c = cell_index(B, ii, jj, p);
        if (sizeof(real) == 4 && a.bfr[0] != nullptr) return a.bfr[d][c];
        return (real)a.bf[d][c];
    };
    // the ring cell of thread t (threads 0 .. NR-1): y rows first (coalesced), then x columns
    auto ring_xy = [&](int& rx, int& ry) {
        if (t < 4 * TX) {
            const int r = t / TX;
            rx = t % TX;
            ry = r < 2 ? r - 2 : TY + r - 2;
        } else {
            const int c = (t - 4 * TX) & 3;
            ry = (t - 4 * TX) >> 2;
            rx = c < 2 ? c - 2 : TX + c - 2;
        }
    };
    real sm = real(0), cfl = real(0);
    real fz[4], dxy[4], dxn[4];   // z flux of the face below; x/y flux differences of the next plane
    real eyx_lo = real(0), eyx_hi = real(0), exy_lo = real(0), exy_hi = real(0);
    real xez = real(0), yez = real(0);       // Ez slots of the x and y face, plane k (then k+1)
    double cz = 0.0, cvx = 0.0, cvy = 0.0;   // centre Ez and velocities, plane k (then k+1)
    double vz_lo = 0.0, vz_hi = 0.0;
    double bz_m = 0.0;
    bool have_bzm = false;
#pragma unroll
    for (int f = 0; f < 4; f++) fz[f] = dxy[f] = dxn[f] = real(0);
    // z march: E and the limited upper state of plane k, and its upper face field
    real Ez_[6], wRz[6], wbz;
    constexpr bool CARRY = sizeof(real) == 4;
    real w0z[CARRY ? 6 : 1], Pn[CARRY ? 7 : 1];   // FP32: the own column's planes k and k+2
    {
        const int tx = (int)(t % TX), ty = (int)(t / TX), i = i0 + tx, j = j0 + ty, own = (ty + 2) * PX + tx + 2;
        real W[4][6], u[7];
        load_cons(i, j, ks - 3, u);
        to_prims(u);
#pragma unroll
        for (int r = 0; r < 6; r++) W[0][r] = u[rslot<2>(r)];
        load_cons(i, j, ks - 2, u);
        to_prims(u);
#pragma unroll
        for (int r = 0; r < 6; r++) W[1][r] = u[rslot<2>(r)];
        load_cons(i, j, ks - 1, u);
        to_prims(u);
#pragma unroll
        for (int f = 0; f < 7; f++) sW[f][own] = u[f];
#pragma unroll
        for (int r = 0; r < 6; r++) W[2][r] = u[rslot<2>(r)];
        load_cons(i, j, ks, u);
        to_prims(u);
#pragma unroll
        for (int r = 0; r < 6; r++) {
            W[3][r] = u[rslot<2>(r)];
            wRz[r] = real(0);
            if constexpr (CARRY) w0z[r] = W[1][r];
        }
        if constexpr (CARRY) {
#pragma unroll
            for (int f = 0; f < 7; f++) Pn[f] = u[f];
        }
        wbz = face_b(2, i, j, ks - 2);
        char_edge(W, wbz, cs, beta, Ez_);
        if (t < NR) {
            int rx, ry;
            ring_xy(rx, ry);
            load_cons(i0 + rx, j0 + ry, ks - 1, u);
            to_prims(u);
#pragma unroll
            for (int f = 0; f < 7; f++) sW[f][(ry + 2) * PX + rx + 2] = u[f];
        }
    }
    __syncthreads();
    // The first pass (k = ks - 2) only forms plane ks - 1, by the same code as every plane.
#pragma unroll 1
    for (int k = ks - 2; k < ke; k++) {
        asm volatile("" : "+v"(lane_bits), "+v"(t));
        const int tx = (int)(t % TX), ty = (int)(t / TX), lane = (int)(t & 63);
        const int i = i0 + tx, j = j0 + ty, own = (ty + 2) * PX + tx + 2;
        const bool live = k >= ks - 1;   // uniform over the workgroup
        const int p = k + 1, q0 = k & 1, q1 = p & 1;
        const bool pt = inr(p, a.ft_lo, n2 + a.ft_hi);
        // ---- A1
        const real wby = face_b(1, i, j, p), wbz1 = face_b(2, i, j, p);
        real P3[7];
        if constexpr (CARRY) load_cons(i, j, k + 3, P3);
        sEf[0][t] = xez;
        sEf[1][t] = yez;
        sV[0][t] = cz;
        sV[1][t] = cvx;
        sV[2][t] = cvy;
        __builtin_amdgcn_sched_barrier(0);
        {   // y
            real W[4][6], E[6];
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int r = 0; r < 6; r++) W[m][r] = sW[rslot<1>(r)][own + (m - 1) * PX];
            char_edge(W, wby, cs, beta, E);
#pragma unroll
            for (int r = 0; r < 6; r++) sEy[r][t + TX] = E[r];
        }
        __builtin_amdgcn_sched_barrier(0);
        if ((int)(t >> 6) == (k & (NW - 1)) && lane < TX + TY) {   // the cells below the tile
            const bool xd = lane >= TX;   // column -1, x direction; else row -1, y direction
            const int ex_ = xd ? -1 : lane, ey_ = xd ? lane - TX : -1;
            const int o = (ey_ + 2) * PX + ex_ + 2, st = xd ? 1 : PX;
            const real wb = xd ? face_b(0, i0 + ex_, j0 + ey_, p) : face_b(1, i0 + ex_, j0 + ey_, p);
            real W[4][6], E[6];
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int r = 0; r < 6; r++) {
                    const int fx = rslot<0>(r), fy = rslot<1>(r);
                    W[m][r] = (&sW[0][0])[(xd ? fx : fy) * (PY * PX) + o + (m - 1) * st];
                }
            char_edge(W, wb, cs, beta, E);
#pragma unroll
            for (int r = 0; r < 6; r++) {
                if (xd) sEx[r][ey_] = E[r];
                else sEy[r][ex_] = E[r];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        {   // z: E of plane k+1, its limited states, face k+1/2
            real W[4][6], E[6], sl[6], sr[6];
            if constexpr (CARRY) {
                to_prims(P3);
#pragma unroll
                for (int r = 0; r < 6; r++) {
                    W[0][r] = w0z[r];
                    W[1][r] = w0z[r] = sW[rslot<2>(r)][own];
                    W[2][r] = Pn[rslot<2>(r)];
                    W[3][r] = P3[rslot<2>(r)];
                }
            } else {
                real P0[7], P2[7];
                load_cons(i, j, k, P0);
                load_cons(i, j, k + 2, P2);
                load_cons(i, j, k + 3, P3);
                to_prims(P0);
                to_prims(P2);
                to_prims(P3);
#pragma unroll
                for (int r = 0; r < 6; r++) {
                    W[0][r] = P0[rslot<2>(r)];
                    W[1][r] = sW[rslot<2>(r)][own];
                    W[2][r] = P2[rslot<2>(r)];
                    W[3][r] = P3[rslot<2>(r)];
                }
            }
            char_edge(W, wbz1, cs, beta, E);
#pragma unroll
            for (int r = 0; r < 6; r++) {
                sl[r] = wRz[r];
                sr[r] = ppm_edge<false>(W[1][r], Ez_[r], E[r]);
                wRz[r] = ppm_edge<true>(W[1][r], Ez_[r], E[r]);
                Ez_[r] = E[r];
            }
            real fu[4] = {real(0), real(0), real(0), real(0)};
            if (live && lb(LB_FZ) && inr(k, a.fn_lo, n2 + a.fn_hi)) {
                real F[7];
                sm = fmax(sm, char_solve<real, RS>(sl, sr, wbz, cs, F));
                fu[0] = F[0]; fu[3] = F[1]; fu[1] = F[2]; fu[2] = F[3];
                sEz3[0][t] = -F[5];
                sEz3[1][t] = F[6];
            } else {
                sEz3[0][t] = sEz3[1][t] = real(0);
            }
            wbz = wbz1;
#pragma unroll
            for (int f = 0; f < 4; f++) {   // the flux divergence of plane k
                dxy[f] = dxy[f] + face_diff(fu[f], fz[f]);
                fz[f] = fu[f];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        vz_hi = 0.0;
        if (lb(LB_CELL) && inr(p, 1 - nb, n2 + nb)) {   // centre EMFs and velocities (FP64) of plane k+1
            real u[7];
            load_cons(i, j, p, u);
            const double r = (double)u[0], m1 = (double)u[1], m2 = (double)u[2], m3 = (double)u[3], b4 = (double)u[4],
                         b5 = (double)u[5], b6 = (double)u[6];
            const double ir = 1.0 / r;
            sC[q1][0][t] = (b5 * m3 - b6 * m2) * ir;
            sC[q1][1][t] = (b6 * m1 - b4 * m3) * ir;
            cz = (b4 * m2 - b5 * m1) * ir;
            if (sizeof(real) == 4) {   // FP32 path: m (1/rho) for the velocities (FP64 keeps the division)
                cvx = m1 * ir;
                cvy = m2 * ir;
                vz_hi = m3 * ir;
            } else {
                cvx = m1 / r;
                cvy = m2 / r;
                vz_hi = m3 / r;
            }
        }
        __syncthreads();
        // ---- A2
        {   // y-face: limited states of the own cell and of the cell above
            real sl[6], sr[6];
#pragma unroll
            for (int r = 0; r < 6; r++) {
                const int f = rslot<1>(r);
                const int tu = ty < TY - 1 ? t + 2 * TX : t + TX;   // row TY-1 forms no face
                const real e0 = sEy[r][t + TX];
                sl[r] = ppm_edge<true>(sW[f][own], sEy[r][t], e0);
                sr[r] = ppm_edge<false>(sW[f][own + PX], e0, sEy[r][tu]);
            }
            if (lb(LB_FY) && pt) {
                real F[7];
                sm = fmax(sm, char_solve<real, RS>(sl, sr, wby, cs, F));
                sF[0][t] = F[0]; sF[2][t] = F[1]; sF[3][t] = F[2]; sF[1][t] = F[3];
                exy_hi = -F[5];
                yez = F[6];
            } else {
                sF[0][t] = sF[1][t] = sF[2][t] = sF[3][t] = real(0);
                exy_hi = yez = real(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        {   // x-face: E of the lane below, limited lower state of the lane above
            real W[4][6], Ex_[6], sl[6], sr[6], fx[4];
            const real wbx = face_b(0, i, j, p);
#pragma unroll
            for (int m = 0; m < 4; m++)
#pragma unroll
                for (int r = 0; r < 6; r++) W[m][r] = sW[rslot<0>(r)][own + m - 1];
            char_edge(W, wbx, cs, beta, Ex_);
#pragma unroll
            for (int r = 0; r < 6; r++) {
                const real below = lane_prev_r(Ex_[r]), edge = sEx[r][ty];
                const real wl = lb(LB_X0) ? edge : below;
                sl[r] = ppm_edge<true>(W[1][r], wl, Ex_[r]);
                sr[r] = lane_next_r(ppm_edge<false>(W[1][r], wl, Ex_[r]));
            }
            if (lb(LB_FX) && pt) {
                real F[7];
                sm = fmax(sm, char_solve<real, RS>(sl, sr, wbx, cs, F));
                fx[0] = F[0]; fx[1] = F[1]; fx[2] = F[2]; fx[3] = F[3];
                xez = -F[5];
                eyx_hi = F[6];
            } else {
                fx[0] = fx[1] = fx[2] = fx[3] = real(0);
                xez = eyx_hi = real(0);
            }
#pragma unroll
            for (int f = 0; f < 4; f++) dxn[f] = face_diff(fx[f], lane_prev_r(fx[f]));
        }
        __syncthreads();
        // ---- D: the update's inputs first, then the corner EMFs of index k, the flux
        // differences of plane k+1 and the primitives of plane k+2
        real div[4];
#pragma unroll
        for (int f = 0; f < 4; f++) div[f] = dxy[f];
        const bool upd = k >= ks && lb(LB_U) && inr(k, a.u_lo, n2 + a.u_hi);
        const bool ccb = lb(LB_CCB) && k >= a.u_lo + sh;
        real w2[7], g[7];
        int rx = 0, ry = 0;
        if constexpr (!CARRY) load_cons(i, j, k + 2, w2);
        if (t < NR) {
            ring_xy(rx, ry);
            load_cons(i0 + rx, j0 + ry, k + 2, g);
        }
        real pq[4] = {real(0), real(0), real(0), real(0)}, pc[4] = {real(0), real(0), real(0), real(0)};
        double pb[3] = {0.0, 0.0, 0.0}, pbm[3] = {0.0, 0.0, 0.0};
        if (upd) {
            const long long c = cell_index(B, i, j, k);
#pragma unroll
            for (int f = 0; f < 4; f++) pq[f] = a.src.q[f][c];
            if (sizeof(real) == 4 && a.comp[0] != nullptr) {
#pragma unroll
                for (int f = 0; f < 4; f++) pc[f] = a.comp[f][c];
            }
#pragma unroll
            for (int d = 0; d < 3; d++) pb[d] = a.src.b[d][c];
            if (ccb) {
                pbm[0] = a.src.b[0][c - sx];
                pbm[1] = a.src.b[1][c - sy];
                if (!have_bzm) pbm[2] = a.src.b[2][c - sz];
            }
        }
        if (live && lb(LB_C) && inr(k, a.c_lo, n2 + a.c_hi)) {
            const double vx = 0.5 * (sV[1][t] + sV[1][t + 1]), vy = 0.5 * (sV[2][t] + sV[2][t + TX]);
            const double vz = 0.5 * (vz_lo + vz_hi);
            double a14, a34, b14, b34;
            {   // Ez at (i+1/2, j+1/2, k); the factor 2 of k_corner's differences taken out
                const double e00 = sV[0][t], e10 = sV[0][t + 1], e01 = sV[0][t + TX], e11 = sV[0][t + TX + 1];
                const double y0 = sEf[1][t], y1 = sEf[1][t + 1], x0 = sEf[0][t], x1 = sEf[0][t + TX];
                upw(vx, y0 - e00, y1 - e10, e01 - y0, e11 - y1, a14, a34);
                upw(vy, x0 - e00, x1 - e01, e10 - x0, e11 - x1, b14, b34);
                sEz[t] = (0.25 * (x0 + x1 + y0 + y1) + 0.25 * ((a14 - a34) + (b14 - b34)));
            }
            {   // Ey at (i+1/2, j, k+1/2)
                const double e00 = sC[q0][1][t], e10 = sC[q0][1][t + 1], e01 = sC[q1][1][t], e11 = sC[q1][1][t + 1];
                const double z0 = sEz3[0][t], z1 = sEz3[0][t + 1], x0 = eyx_lo, x1 = eyx_hi;
                upw(vx, z0 - e00, z1 - e10, e01 - z0, e11 - z1, a14, a34);
                upw(vz, x0 - e00, x1 - e01, e10 - x0, e11 - x1, b14, b34);
                sEc[q0][1][t] = (0.25 * (x0 + x1 + z0 + z1) + 0.25 * ((a14 - a34) + (b14 - b34)));
            }
            {   // Ex at (i, j+1/2, k+1/2)
                const double e00 = sC[q0][0][t], e10 = sC[q0][0][t + TX], e01 = sC[q1][0][t], e11 = sC[q1][0][t + TX];
                const double z0 = sEz3[1][t], z1 = sEz3[1][t + TX], y0 = exy_lo, y1 = exy_hi;
                upw(vy, z0 - e00, z1 - e10, e01 - z0, e11 - z1, a14, a34);
                upw(vz, y0 - e00, y1 - e01, e10 - y0, e11 - y1, b14, b34);
                sEc[q0][0][t] = (0.25 * (y0 + y1 + z0 + z1) + 0.25 * ((a14 - a34) + (b14 - b34)));
            }
        }
        if constexpr (CARRY) {
#pragma unroll
            for (int f = 0; f < 7; f++) {
                sW[f][own] = Pn[f];
                Pn[f] = P3[f];
            }
        } else {
            to_prims(w2);
#pragma unroll
            for (int f = 0; f < 7; f++) sW[f][own] = w2[f];
        }
        if (t < NR) {
            to_prims(g);
#pragma unroll
            for (int f = 0; f < 7; f++) sW[f][(ry + 2) * PX + rx + 2] = g[f];
        }
        if (lb(LB_U)) {
#pragma unroll
            for (int f = 0; f < 4; f++) dxy[f] = dxn[f] + (sF[f][t] - sF[f][t - TX]);
        }
        __syncthreads();
        // ---- G: update of plane k (k_update_z's arithmetic)
        if (upd) {
            const long long c = cell_index(B, i, j, k);
            real nq[7], oq[4];
#pragma unroll
            for (int f = 0; f < 4; f++) {
                const real q0v = pq[f];
                oq[f] = q0v;
                real v;
                if (sizeof(real) == 4 && a.comp[0] != nullptr) {   // Kahan terms
                    const real y = -(dtdx * div[f]) - pc[f];
                    v = q0v + y;
                    a.comp[f][c] = (v - q0v) - y;
                } else {
                    v = q0v - dtdx * div[f];
                }
                if (f == 0 && v < (real)MIN_DENS) {
                    v = (real)MIN_DENS;
                    if (sizeof(real) == 4 && a.comp[0] != nullptr) a.comp[0][c] = real(0);
                    atomicAdd(a.floor_count, a.img ? floor_images(n0, n1, n2, i, j, k, a.img_lo, a.img_hi) : 1u);
                }
                a.dst.q[f][c] = v;
                nq[f] = v;
            }
            const double ex = sEc[q0][0][t], ey = sEc[q0][1][t], ez = sEz[t];
            const double ez_y = sEz[t - TX], ez_x = sEz[t - 1], ey_x = sEc[q0][1][t - 1], ex_y = sEc[q0][0][t - TX];
            const double ex_m = sEc[q1][0][t], ey_m = sEc[q1][1][t], eyx_m = sEc[q1][1][t - 1], exy_m = sEc[q1][0][t - TX];
            const double bx = pb[0] - dtd * ((ez - ez_y) - (ey - ey_m));
            const double by = pb[1] - dtd * ((ex - ex_m) - (ez - ez_x));
            const double bz = pb[2] - dtd * ((ey - ey_x) - (ex - ex_y));
            a.dst.b[0][c] = bx;
            a.dst.b[1][c] = by;
            a.dst.b[2][c] = bz;
            if (ccb) {
                const double ez_xy = sEz[t - 1 - TX];
                const double bxm = pbm[0] - dtd * ((ez_x - ez_xy) - (ey_x - eyx_m));
                const double bym = pbm[1] - dtd * ((ex_y - exy_m) - (ez_y - ez_xy));
                if (!have_bzm) bz_m = pbm[2] - dtd * ((ey_m - eyx_m) - (ex_m - exy_m));
                nq[4] = (real)(0.5 * (bx + bxm));
                nq[5] = (real)(0.5 * (by + bym));
                nq[6] = (real)(0.5 * (bz + bz_m));
            } else {
#pragma unroll
                for (int f = 4; f < 7; f++) nq[f] = a.src.q[f][c];
            }
#pragma unroll
            for (int f = 4; f < 7; f++) a.dst.q[f][c] = nq[f];
            bz_m = bz;
            have_bzm = true;
            if (a.pvel[0] != nullptr) {   // passive velocities (copy_velocity's arithmetic)
                const real io = fdiv(real(1), oq[0]), in = fdiv(real(1), nq[0]);
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const real vo = oq[1 + d] * io;
                    a.pvel[d][c] = real(0.5) * (vo + nq[1 + d] * in);
                }
            }
            if (a.cmax != nullptr && lb(LB_INT) && k >= 1 && k <= n2) {
                if constexpr (sizeof(real) == 4) cfl = fmax(cfl, cell_fast_speed_f(nq, (float)a.cs));
                else cfl = fmax(cfl, cell_fast_speed(nq, a.cs));
            }
        } else {
            have_bzm = false;
        }
        eyx_lo = eyx_hi;
        exy_lo = exy_hi;
        vz_lo = vz_hi;
    }
    atomic_max_nonneg(a.smax, b, (double)sm);
    if (a.cmax != nullptr) atomic_max_nonneg(a.cmax, b, (double)cfl);
}

template <class real, int RS, class F>
auto vl_char_shape(int shape, F f) {
    if (shape == 0) return f(k_vl_char<real, RS, vs_tx(0), vs_ty(0)>, vs_tx(0) * vs_ty(0));
    return f(k_vl_char<real, RS, vs_tx(1), vs_ty(1)>, vs_tx(1) * vs_ty(1));
}
template <class real, int RS>
void launch_vl_char(hipStream_t st, const BoxDesc* boxes, const TilePlan& plan, const StageArgs<real>& a, int shape) {
    if (plan.total <= 0) return;
    vl_char_shape<real, RS>(shape, [&](auto kern, int n) {
        hipLaunchKernelGGL(kern, dim3((unsigned)plan.total), dim3(n), 0, st, boxes, plan, a);
    });
}
template <class real, int RS>
int vl_char_blocks_per_cu(int shape) {
    return vl_char_shape<real, RS>(shape, [&](auto kern, int nt) {
        int n = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, nt, 0);
        return e == hipSuccess && n > 0 ? n : 1;
    });
}

#define IMHD_INST_CHAR(real, RS)                                                                                          \
    template void launch_vl_char<real, RS>(hipStream_t, const BoxDesc*, const TilePlan&, const StageArgs<real>&, int); \
    template int vl_char_blocks_per_cu<real, RS>(int);

}  // namespace imhd
