// Power spectra and density PDF of the reference's analysis program
// (3D_MPI/Analysis/src/analysis_main.f90:105-226, 543-698) on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include "spectra.hpp"

namespace imhd {

// The REAL*4 components of the analysed field on the interior, as the analysis program forms
// them from the snapshot: v = (rho v)/rho; v_par = (v.B/|B|) B/|B|; v_perp = v - v_par.
// Bound by memory: all requested components from one read of the fields that they need
// (FP32 256^3: three components of v_perp in 0.12 ms; one launch per component, each reading
// all seven fields behind 64-bit index divisions, took 0.31).
template <class real, int WHICH>
__global__ __launch_bounds__(256) void k_spec_pack(BoxDesc B, SpecPackArgs<real> a) {
    const long long g0 = (long long)blockIdx.x * 256, g = g0 + threadIdx.x;
    if (g >= (long long)B.n[0] * B.n[1] * B.n[2]) return;
    unsigned i, j, k;
    item_xyz((unsigned long long)g0, threadIdx.x, (unsigned)B.n[0], (unsigned)B.n[1], i, j, k);
    const long long c = cell_index(B, (int)i + 1, (int)j + 1, (int)k + 1);
    if (WHICH == SPEC_DENSITY) {
        a.out[0][g] = (float)a.q[0][c];
        return;
    }
    const bool full = WHICH == SPEC_VPAR || WHICH == SPEC_VPERP;
    float f[7];
#pragma unroll
    for (int m = 0; m < 7; m++)
        if (full || (WHICH == SPEC_VELOCITY && (m == 0 || (m < 4 && a.out[m - 1]))) ||
            (WHICH == SPEC_BFIELD && m >= 4 && a.out[m - 4]))
            f[m] = (float)a.q[m][c];
    float bmag = 0.0f, vdotb = 0.0f;
    if (full) {
        bmag = sqrtf(f[4] * f[4] + f[5] * f[5] + f[6] * f[6]);
        vdotb = (f[1] / f[0] * f[4] + f[2] / f[0] * f[5] + f[3] / f[0] * f[6]) / bmag;
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        if (!a.out[d]) continue;
        float out;
        if (WHICH == SPEC_BFIELD) out = f[4 + d];
        else if (WHICH == SPEC_VELOCITY) out = f[1 + d] / f[0];
        else if (WHICH == SPEC_VPAR) out = vdotb * (f[4 + d] / bmag);
        else out = f[1 + d] / f[0] - vdotb * (f[4 + d] / bmag);
        a.out[d][g] = out;
    }
}

__global__ __launch_bounds__(256) void k_spec_accum(const float* __restrict__ F, int n, float* __restrict__ s,
                                                    int first) {
    const int h = n / 2;
    const long long g0 = (long long)blockIdx.x * 256, g = g0 + threadIdx.x;
    if (g >= (long long)h * h * h) return;
    unsigned kx, ky, kz;
    item_xyz((unsigned long long)g0, threadIdx.x, (unsigned)h, (unsigned)h, kx, ky, kz);
    const long long o = ((long long)kz * n + ky) * (h + 1) + kx;   // R2C output [z][y][x/2+1]
    const float re = F[2 * o], im = F[2 * o + 1];
    float acc = first ? 0.0f : s[g];
    acc = acc + re * re;
    acc = acc + im * im;
    s[g] = acc;
}

// Histogram of a workgroup's run of modes in LDS (n <= SPEC_MAXBINS), then one global add per
// bin.  At most SPEC_BLOCKS workgroups, with runs of modes as long as that takes: every
// workgroup's add to a bin waits for the one before it (about 12 ns), and at one workgroup per
// 256 modes these chains were the kernel's time (256^3: 142 us, 19 in 512 workgroups).
constexpr int SPEC_MAXBINS = 4096;
constexpr int SPEC_BLOCKS = 512;

// Items [first, last) of this workgroup: runs of whole 256s, as even as they come
__device__ __forceinline__ void block_run(long long n, long long& first, long long& last) {
    const long long per = ((n + 255) / 256 + gridDim.x - 1) / gridDim.x * 256;
    first = per * blockIdx.x;
    last = first + per < n ? first + per : n;
}

__global__ __launch_bounds__(256) void k_spec_bin(const float* __restrict__ s, int n, float k0, float dk,
                                                  double* __restrict__ pk) {
    extern __shared__ double spec_hist[];
    double* hist = spec_hist;
    for (int b = threadIdx.x; b < n; b += 256) hist[b] = 0.0;
    __syncthreads();
    const int h = n / 2;
    long long first, last;
    block_run((long long)h * h * h, first, last);
    for (long long g0 = first; g0 < last; g0 += 256) {
        const long long g = g0 + threadIdx.x;
        if (g >= last) break;
        unsigned kx, ky, kz;
        item_xyz((unsigned long long)g0, threadIdx.x, (unsigned)h, (unsigned)h, kx, ky, kz);
        float fk = 2.0f * s[g];
        if (g == 0) fk = 0.5f * fk;
        const float k = k0 * sqrtf((float)(int)(kx * kx + ky * ky + kz * kz));
        const int ik = (int)(k / dk);
        if (ik >= 0 && ik < n) atomicAdd(&hist[ik], (double)fk);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < n; b += 256)
        if (hist[b] != 0.0) atomicAdd(&pk[b], hist[b]);
}

// Density histogram.  A narrow distribution (a nearly uniform density puts every cell in
// one bin) must not serialise on one counter, so the lanes that share the first pending
// lane's bin are counted by ballot and added once.  With the counts in LDS (nbins <=
// HIST_LDS_BINS) the other lanes then add for themselves, which the LDS serialises only
// among equal bins (a ballot per distinct bin of the wave, up to 64 in turn, made a broad
// distribution 149 us at 256^3 FP32, 63 so; few populated bins are no slower either: a call
// with 2 to 4 takes 85 to 89 us, 101 to 111 with a ballot each); straight into the global
// counts, for more bins, every distinct bin has its ballot.  Counts are exact integers, so the
// order does not matter.
constexpr int HIST_LDS_BINS = 4096;
template <class real, bool LDS>
__global__ __launch_bounds__(256) void k_density_hist(BoxDesc B, const real* __restrict__ rho, float drho, int nbins,
                                                      unsigned long long* __restrict__ counts) {
    __shared__ unsigned int sh[LDS ? HIST_LDS_BINS : 1];
    if (LDS) {
        for (int b = threadIdx.x; b < nbins; b += 256) sh[b] = 0u;
        __syncthreads();
    }
    const long long n = (long long)B.n[0] * B.n[1] * B.n[2];
    const int lane = threadIdx.x & 63;
    long long first, last;
    block_run(n, first, last);
    // the trip count depends on the block only, so every lane of a wave takes part in
    // every ballot
    for (long long g0 = first; g0 < last; g0 += 256) {
        int ib = -1;
        if (g0 + threadIdx.x < last) {
            unsigned i, j, k;
            item_xyz((unsigned long long)g0, threadIdx.x, (unsigned)B.n[0], (unsigned)B.n[1], i, j, k);
            const float r = (float)rho[cell_index(B, (int)i + 1, (int)j + 1, (int)k + 1)];
            const float x = r / drho;
            if (x >= 0.0f) {
                const int v = (int)x;
                if (v < nbins) ib = v;
            }
        }
        bool pending = ib >= 0;
        while (true) {
            const unsigned long long m = __ballot(pending);
            if (m == 0ull) break;
            const int leader = __ffsll((long long)m) - 1;
            const int bin = __shfl(ib, leader);
            const bool mine = pending && ib == bin;
            const unsigned long long same = __ballot(mine);
            if (lane == leader) {
                if (LDS) atomicAdd(&sh[bin], (unsigned int)__popcll(same));
                else atomicAdd(&counts[bin], (unsigned long long)__popcll(same));
            }
            if (mine) pending = false;
            if (LDS) {
                if (pending) atomicAdd(&sh[ib], 1u);
                break;
            }
        }
    }
    if (LDS) {
        __syncthreads();
        for (int b = threadIdx.x; b < nbins; b += 256)
            if (sh[b]) atomicAdd(&counts[b], (unsigned long long)sh[b]);
    }
}

// Sums of B over the interior.  One workgroup per CU, each over a run of cells, with one add
// per component at the end: an add waits for the one before it, and one per 256 cells
// (196608 at 256^3) took 2.36 ms, against 0.056 now, which is the read of the three fields.
constexpr int MEANB_BLOCKS = 256, MEANB_THREADS = 1024;
template <class real>
__global__ __launch_bounds__(MEANB_THREADS) void k_mean_b(BoxDesc B, const real* __restrict__ bx,
                                                          const real* __restrict__ by, const real* __restrict__ bz,
                                                          double* __restrict__ sum) {
    __shared__ double sh[3][MEANB_THREADS / 64];
    const long long rows = (long long)B.n[1] * B.n[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n0 = B.n[0];
    double v[3] = {0.0, 0.0, 0.0};
    // a wave sums whole rows
    for (long long row = (long long)blockIdx.x * (MEANB_THREADS / 64) + wave; row < rows;
         row += (long long)gridDim.x * (MEANB_THREADS / 64)) {
        const int k = (int)(row / B.n[1]), j = (int)(row - (long long)k * B.n[1]);
        const long long c = cell_index(B, 1, j + 1, k + 1);
#pragma unroll 4
        for (int i = lane; i < n0; i += 64) {
            v[0] += (double)(float)bx[c + i];
            v[1] += (double)(float)by[c + i];
            v[2] += (double)(float)bz[c + i];
        }
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        for (int o = 32; o > 0; o >>= 1) v[d] += __shfl_down(v[d], o);
        if (lane == 0) sh[d][wave] = v[d];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double s = 0.0;
        for (int w = 0; w < MEANB_THREADS / 64; w++) s += sh[threadIdx.x][w];
        atomicAdd(&sum[threadIdx.x], s);
    }
}

// One octant mode of mode_decomposition (analysis_main.f90:362-527).  The geometry is
// evaluated in FP64.
constexpr int MODE_LDS_BINS = 512;

template <bool LDS>
__global__ __launch_bounds__(256) void k_mode_bin(const float* __restrict__ F0, const float* __restrict__ F1,
                                                  const float* __restrict__ F2, int n, const double* __restrict__ b0sum,
                                                  float k0f, float dkf, double* __restrict__ P) {
    __shared__ double hist[LDS ? 8 * MODE_LDS_BINS : 1];
    if (LDS) {
        for (int b = threadIdx.x; b < 8 * n; b += 256) hist[b] = 0.0;
        __syncthreads();
    }
    const int h = n / 2;
    const double nc = (double)n * n * n;
    const double B0[3] = {b0sum[0] / nc, b0sum[1] / nc, b0sum[2] / nc};
    const double bsq = B0[0] * B0[0] + B0[1] * B0[1] + B0[2] * B0[2];
    const double bmag = sqrt(bsq), alpha = 1.0 / bsq;
    const double ph[3] = {B0[0] / bmag, B0[1] / bmag, B0[2] / bmag};
    const double k0 = (double)k0f;
    long long first, last;
    block_run((long long)h * h * h, first, last);
    for (long long g0 = first; g0 < last; g0 += 256) {
        const long long g = g0 + threadIdx.x;
        if (g >= last) break;
        if (g == 0) continue;
        unsigned ux, uy, uz;
        item_xyz((unsigned long long)g0, threadIdx.x, (unsigned)h, (unsigned)h, ux, uy, uz);
        const int kx = (int)ux, ky = (int)uy, kz = (int)uz;
        double amp[8];
        const double kv[3] = {k0 * kx, k0 * ky, k0 * kz};
        const double k = k0 * sqrt((double)(kx * kx + ky * ky + kz * kz));
        const double khat[3] = {kv[0] / k, kv[1] / k, kv[2] / k};
        const double kd = kv[0] * ph[0] + kv[1] * ph[1] + kv[2] * ph[2];
        double kpar[3], kperp[3], kph[3] = {0.0, 0.0, 0.0};
        for (int d = 0; d < 3; d++) { kpar[d] = kd * ph[d]; kperp[d] = kv[d] - kpar[d]; }
        const double kpn = sqrt(kperp[0] * kperp[0] + kperp[1] * kperp[1] + kperp[2] * kperp[2]);
        if (kpn > 0.0) for (int d = 0; d < 3; d++) kph[d] = kperp[d] / kpn;
        const double kpar2 = kpar[0] * kpar[0] + kpar[1] * kpar[1] + kpar[2] * kpar[2];
        const double D = fmax(0.0, (1.0 + alpha) * (1.0 + alpha) - 4.0 * alpha * kpar2 / (k * k));
        const double sD = sqrt(D);
        const double za[3] = {kph[1] * ph[2] - kph[2] * ph[1], kph[2] * ph[0] - kph[0] * ph[2],
                              kph[0] * ph[1] - kph[1] * ph[0]};
        double zf[3], zs[3];
        for (int d = 0; d < 3; d++) {
            zf[d] = (-1.0 + alpha + sD) * kpar[d] + (1.0 + alpha + sD) * kperp[d];
            zs[d] = (-1.0 + alpha - sD) * kpar[d] + (1.0 + alpha - sD) * kperp[d];
        }
        const double nf = sqrt(zf[0] * zf[0] + zf[1] * zf[1] + zf[2] * zf[2]);
        const double ns = sqrt(zs[0] * zs[0] + zs[1] * zs[1] + zs[2] * zs[2]);
        if (nf > 0.0) for (int d = 0; d < 3; d++) zf[d] /= nf;
        if (ns > 0.0) for (int d = 0; d < 3; d++) zs[d] /= ns;
        const long long o = ((long long)kz * n + ky) * (h + 1) + kx;
        const double fr[3] = {F0[2 * o], F1[2 * o], F2[2 * o]};
        const double fi[3] = {F0[2 * o + 1], F1[2 * o + 1], F2[2 * o + 1]};
        double va[2] = {0, 0}, vf[2] = {0, 0}, vs[2] = {0, 0};
        for (int d = 0; d < 3; d++) {
            va[0] += fr[d] * za[d]; va[1] += fi[d] * za[d];
            vf[0] += fr[d] * zf[d]; vf[1] += fi[d] * zf[d];
            vs[0] += fr[d] * zs[d]; vs[1] += fi[d] * zs[d];
        }
        const double cf = sqrt(0.5 * bsq * (1.0 + alpha + sD));
        const double csl = sqrt(fmax(0.0, 0.5 * bsq * (1.0 + alpha - sD)));
        const double t1 = khat[0] * zf[0] + khat[1] * zf[1] + khat[2] * zf[2];
        const double t2 = khat[0] * zs[0] + khat[1] * zs[1] + khat[2] * zs[2];
        const double dvf = 2.0 * vf[1], dvs = 2.0 * vs[1];
        auto cross_norm = [&](const double* z) {
            const double c0 = B0[1] * z[2] - B0[2] * z[1], c1 = B0[2] * z[0] - B0[0] * z[2],
                         c2 = B0[0] * z[1] - B0[1] * z[0];
            return sqrt(c0 * c0 + c1 * c1 + c2 * c2);
        };
        // a zero slow speed (k along B0) leaves the reference's slow density and field
        // amplitudes undefined (0/0); they are not counted here
        const double rf = dvf * t1 / cf, rs = csl > 0.0 ? dvs * t2 / csl : 0.0;
        const double bf = dvf * cross_norm(zf) / cf, bs = csl > 0.0 ? dvs * cross_norm(zs) / csl : 0.0;
        amp[0] = 2.0 * (va[0] * va[0] + va[1] * va[1]);
        amp[1] = 2.0 * (vf[0] * vf[0] + vf[1] * vf[1]);
        amp[2] = 2.0 * (vs[0] * vs[0] + vs[1] * vs[1]);
        amp[3] = amp[0];
        amp[4] = 2.0 * bf * bf;
        amp[5] = 2.0 * bs * bs;
        amp[6] = 2.0 * rf * rf;
        amp[7] = 2.0 * rs * rs;
        const float kf = k0f * sqrtf((float)(kx * kx + ky * ky + kz * kz));
        const int ik = (int)(kf / dkf);
        if (ik < 0 || ik >= n) continue;
#pragma unroll
        for (int m = 0; m < 8; m++) atomicAdd(LDS ? &hist[m * n + ik] : &P[m * n + ik], amp[m]);
    }
    if (LDS) {
        __syncthreads();
        for (int b = threadIdx.x; b < 8 * n; b += 256)
            if (hist[b] != 0.0) atomicAdd(&P[b], hist[b]);
    }
}

template <class real>
void launch_mean_b(hipStream_t st, const BoxDesc& B, const real* bx, const real* by, const real* bz, double* sum) {
    const long long rows = (long long)B.n[1] * B.n[2], waves = MEANB_THREADS / 64;
    const unsigned blocks = (unsigned)std::min<long long>((rows + waves - 1) / waves, MEANB_BLOCKS);
    hipLaunchKernelGGL((k_mean_b<real>), dim3(blocks), dim3(MEANB_THREADS), 0, st, B, bx, by, bz, sum);
}
void launch_mode_bin(hipStream_t st, const float* F0, const float* F1, const float* F2, int n, const double* b0sum,
                     float k0, float dk, double* P) {
    const long long m = (long long)(n / 2) * (n / 2) * (n / 2);
    // past MODE_LDS_BINS every mode adds to the global sums, and more workgroups do not add
    // more; within it, 1024 workgroups (four waves per SIMD) and their chains of adds
    const dim3 grid((unsigned)std::min<long long>((m + 255) / 256, n <= MODE_LDS_BINS ? 1024 : 65536));
    if (n <= MODE_LDS_BINS)
        hipLaunchKernelGGL(k_mode_bin<true>, grid, dim3(256), 0, st, F0, F1, F2, n, b0sum, k0, dk, P);
    else
        hipLaunchKernelGGL(k_mode_bin<false>, grid, dim3(256), 0, st, F0, F1, F2, n, b0sum, k0, dk, P);
}

template <class real>
void launch_spec_pack(hipStream_t st, const BoxDesc& B, const SpecPackArgs<real>& a) {
    const long long n = (long long)B.n[0] * B.n[1] * B.n[2];
    const dim3 grid((unsigned)((n + 255) / 256));
    switch (a.which) {
        case SPEC_DENSITY: hipLaunchKernelGGL((k_spec_pack<real, SPEC_DENSITY>), grid, dim3(256), 0, st, B, a); break;
        case SPEC_VELOCITY: hipLaunchKernelGGL((k_spec_pack<real, SPEC_VELOCITY>), grid, dim3(256), 0, st, B, a); break;
        case SPEC_BFIELD: hipLaunchKernelGGL((k_spec_pack<real, SPEC_BFIELD>), grid, dim3(256), 0, st, B, a); break;
        case SPEC_VPAR: hipLaunchKernelGGL((k_spec_pack<real, SPEC_VPAR>), grid, dim3(256), 0, st, B, a); break;
        default: hipLaunchKernelGGL((k_spec_pack<real, SPEC_VPERP>), grid, dim3(256), 0, st, B, a);
    }
}
void launch_spec_accum(hipStream_t st, const float* F, int n, float* s, int first) {
    const long long m = (long long)(n / 2) * (n / 2) * (n / 2);
    hipLaunchKernelGGL(k_spec_accum, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, F, n, s, first);
}
void launch_spec_bin(hipStream_t st, const float* s, int n, float k0, float dk, double* pk) {
    const long long m = (long long)(n / 2) * (n / 2) * (n / 2);
    const unsigned blocks = (unsigned)std::min<long long>((m + 255) / 256, SPEC_BLOCKS);
    hipLaunchKernelGGL(k_spec_bin, dim3(blocks), dim3(256), (size_t)n * 8, st, s, n, k0, dk, pk);
}
template <class real>
void launch_density_hist(hipStream_t st, const BoxDesc& B, const real* rho, float drho, int nbins,
                         unsigned long long* counts) {
    const long long n = (long long)B.n[0] * B.n[1] * B.n[2];
    const unsigned blocks = (unsigned)std::min<long long>((n + 255) / 256, 2048);
    if (nbins <= HIST_LDS_BINS)
        hipLaunchKernelGGL((k_density_hist<real, true>), dim3(blocks), dim3(256), 0, st, B, rho, drho, nbins, counts);
    else
        hipLaunchKernelGGL((k_density_hist<real, false>), dim3(blocks), dim3(256), 0, st, B, rho, drho, nbins, counts);
}

template void launch_spec_pack<double>(hipStream_t, const BoxDesc&, const SpecPackArgs<double>&);
template void launch_spec_pack<float>(hipStream_t, const BoxDesc&, const SpecPackArgs<float>&);
template void launch_mean_b<double>(hipStream_t, const BoxDesc&, const double*, const double*, const double*, double*);
template void launch_mean_b<float>(hipStream_t, const BoxDesc&, const float*, const float*, const float*, double*);
template void launch_density_hist<double>(hipStream_t, const BoxDesc&, const double*, float, int,
                                          unsigned long long*);
template void launch_density_hist<float>(hipStream_t, const BoxDesc&, const float*, float, int, unsigned long long*);

}  // namespace imhd
