// rl2_kernels.hip -- gfx950 kernels of the per-galaxy shape-measurement path.
//
// Residual layout: channel-major R[c * nrow + i] over rows i in the observation's
// spatially sorted order (Morton order of (u, v)), complex128 (RL2_PREC_FP64) or
// complex64 (RL2_PREC_MIXED).  sigma^2 is one float per visibility with the sign bit
// marking a flagged visibility (sigma^2 > 0 after defaulting, RadioLensfit2.cpp:266-269).
#include <hip/hip_runtime.h>
#include <map>

#include <algorithm>
#include <cmath>
#include <hipcub/hipcub.hpp>

#include "rl2_internal.h"
#include "rl2_gk41.h"

namespace rl2 {

constexpr uint32_t kEmpty = 0xffffffffu;

// ------------------------------------------------------------------ small helpers
__device__ inline double2 load_res(const void *res, int prec, size_t k)
{
    if (prec == 0) return reinterpret_cast<const double2 *>(res)[k];
    float2 f = reinterpret_cast<const float2 *>(res)[k];
    return make_double2((double)f.x, (double)f.y);
}
__device__ inline void store_res(void *res, int prec, size_t k, double2 v)
{
    if (prec == 0)
        reinterpret_cast<double2 *>(res)[k] = v;
    else
        reinterpret_cast<float2 *>(res)[k] = make_float2((float)v.x, (float)v.y);
}

// Round-model / fitted-model visibility of one galaxy in one channel at one row
// (galaxy_visibilities.c:154-190), returned with its phase rotor.
__device__ inline double model_shape(const GalaxyGeom &g, double u, double v, double wn2,
                                     double spectra)
{
    double k1 = (1. + g.e1) * u + g.e2 * v;
    double k2 = g.e2 * u + (1. - g.e1) * v;
    double shape = sersic_shape(k1, k2, g.sf, wn2);
    return shape * (spectra * g.flux);
}

// 1 / sqrt(a) for a >= 1: the hardware estimate refined once, r + r e (1/2 + 3/8 e) with
// e = 1 - a r^2 (bit-identical to rsqrt(), which adds a class test of the estimate for
// zero, infinite and denormal arguments that a >= 1 never has).
__device__ inline double rsqrt_ge1(double a)
{
    const double r = __builtin_amdgcn_rsq(a);
    const double e = fma(-a * r, r, 1.);
    return fma(r * e, fma(e, 0.375, 0.5), r);
}

// The same model with (1 + s w |k|^2)^(-3/2) as rsqrt(den)^3 (one reciprocal square
// root instead of a square root and a division; a few ulp from the reference's form).
// model_kk: |k|^2 of a row, the same in all its channels.
__device__ inline double model_kk(const GalaxyGeom &g, double u, double v)
{
    const double k1 = fma(g.e2, v, (1. + g.e1) * u);
    const double k2 = fma(1. - g.e1, v, g.e2 * u);
    return fma(k1, k1, k2 * k2);
}
__device__ inline double model_shape_kk(const GalaxyGeom &g, double kk, double wn2, double spectra)
{
    const double rr = rsqrt_ge1(fma(g.sf * wn2, kk, 1.));
    return rr * rr * rr * (spectra * g.flux);
}
__device__ inline double model_shape_rsq(const GalaxyGeom &g, double u, double v, double wn2,
                                         double spectra)
{
    return model_shape_kk(g, model_kk(g, u, v), wn2, spectra);
}
// For any galaxy a caller may name: an ellipticity on the unit circle, or a scalelength without a
// finite square, has an infinite denominator a and the model 0 (as 1 / (a sqrt(a)) gives it); a
// NaN stays one (the estimate's).  a^(-3/2) is formed from the hardware's estimate r directly,
// r^3 (1 + 3/2 e + 15/8 e^2) with e = 1 - a r^2 to twice the precision: two roundings, where the
// cube of a rounded reciprocal root carries three of the root's.
__device__ inline double model_shape_any(const GalaxyGeom &g, double u, double v, double wn2,
                                         double spectra)
{
    const double a = fma(g.sf * wn2, model_kk(g, u, v), 1.);
    const double r = __builtin_amdgcn_rsq(a), b = fmin(a, 1.7976931348623157e308);
    const double h = r * r, hl = fma(r, r, -h), r3 = h * r;
    const double e = fma(-b, hl, fma(-b, h, 1.));
    return fma(r3 * e, fma(e, 1.875, 1.5), r3) * (spectra * g.flux);
}

// One visibility of the post-fit update (data_processing.c:109-135): R = (R - fit) + round,
// both models with the phase rotor of the fitted galaxy's position (p = u l + v m + w n,
// the phase k p in revolutions is p / lambda).
__device__ inline double2 subtract_vis_kk(const GalaxyGeom &fit, const GalaxyGeom &rnd, double p,
                                          double kk_fit, double kk_rnd, double k2, double spectra,
                                          double inv_lambda, double2 r)
{
    double sn, cs;
    sincos_rev64(p * inv_lambda, sn, cs);
    const double sr = model_shape_kk(rnd, kk_rnd, k2, spectra);
    const double sfit = model_shape_kk(fit, kk_fit, k2, spectra);
    r.x = (r.x - sfit * cs) + sr * cs;
    r.y = (r.y - sfit * sn) + sr * sn;
    return r;
}

__device__ inline double2 subtract_vis(const GalaxyGeom &fit, const GalaxyGeom &rnd, double p,
                                       double u, double v, double k2, double spectra,
                                       double inv_lambda, double2 r)
{
    return subtract_vis_kk(fit, rnd, p, model_kk(fit, u, v), model_kk(rnd, u, v), k2, spectra,
                           inv_lambda, r);
}

// ------------------------------------------------------------------ sources / noise
// R += sign * sum_g flux_g spec_c shape_g exp(i k_c (u l + v m + w n)).
// One thread per row; galaxies staged through LDS in tiles of 128.
// Bound by FP64 issue (a phase and a model per galaxy and visibility, about 60 FP64 and integer
// instructions), so the phase goes through sincos_rev_near and the model through one reciprocal
// square root, and whole blocks of CB channels run without a test per channel.  500 galaxies
// on 3.87M visibilities: 3.4 ms; 6.1 with the library's sincos and a square root and a division
// per model.  The error against 80 bits is 0.87 of that form's (2.0e-15 against 2.3e-15 of the
// model, rms, on phases of up to 40 revolutions; 0.92 of it in the modulus).
template <int PREC, int CB>
__device__ inline void add_sources_block(const GalaxyGeom *__restrict__ gal, unsigned ngal,
                                         unsigned c0, unsigned long nrow, unsigned long i,
                                         double ui, double vi, double wi,
                                         const double *__restrict__ wn,
                                         const double *__restrict__ inv_lambda,
                                         const double *__restrict__ spec, double sign, void *res)
{
    constexpr int TILE = 128;
    __shared__ GalaxyGeom sg[TILE];
    // what 1 / lambda lacks of k / (2 pi): the phase then carries no rounding but that of p, where
    // the product k p carries its own (1 / lambda alone would add two)
    constexpr double kTwoPiLo = 2.4492935982947064e-16;
    double are[CB], aim[CB], il_lo[CB];
#pragma unroll
    for (int k = 0; k < CB; k++) {
        are[k] = aim[k] = 0.;
        const double il = inv_lambda[c0 + k];
        il_lo[k] = (fma(-il, kTwoPi, wn[c0 + k]) - il * kTwoPiLo) * (1. / kTwoPi);
    }
    for (unsigned g0 = 0; g0 < ngal; g0 += TILE) {
        __syncthreads();
        for (unsigned t = threadIdx.x; t < TILE && g0 + t < ngal; t += blockDim.x)
            sg[t] = gal[g0 + t];
        __syncthreads();
        const unsigned gn = min((unsigned)TILE, ngal - g0);
        for (unsigned t = 0; t < gn; t++) {
            const GalaxyGeom g = sg[t];
            const double p = ui * g.l0 + vi * g.m0 + wi * g.n0;
#pragma unroll
            for (int k = 0; k < CB; k++) {
                // the phase k p in revolutions is p / lambda
                const double wnc = wn[c0 + k];
                const double shape = model_shape_any(g, ui, vi, wnc * wnc, spec[c0 + k]);
                const double il = inv_lambda[c0 + k], t = p * il;
                double sn, cs;
                sincos_rev_near((t - rint(t)) + fma(p, il_lo[k], fma(p, il, -t)), sn, cs);
                are[k] = fma(shape, cs, are[k]);
                aim[k] = fma(shape, sn, aim[k]);
            }
        }
    }
    if (i >= nrow) return;
#pragma unroll
    for (int k = 0; k < CB; k++) {
        const size_t idx = (size_t)(c0 + k) * nrow + i;
        double2 r = load_res(res, PREC, idx);
        r.x += sign * are[k];
        r.y += sign * aim[k];
        store_res(res, PREC, idx, r);
    }
}

template <int PREC>
__global__ __launch_bounds__(256) void add_sources_kernel(unsigned nch, unsigned long nrow,
                                                          const double *__restrict__ u,
                                                          const double *__restrict__ v,
                                                          const double *__restrict__ w,
                                                          const double *__restrict__ wn,
                                                          const double *__restrict__ inv_lambda,
                                                          const double *__restrict__ spec,
                                                          const GalaxyGeom *__restrict__ gal,
                                                          unsigned ngal, double sign, void *res)
{
    const unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    const bool ok = i < nrow;
    const double ui = ok ? u[i] : 0., vi = ok ? v[i] : 0., wi = ok ? w[i] : 0.;
    unsigned c0 = 0;
    for (; c0 + 4 <= nch; c0 += 4)
        add_sources_block<PREC, 4>(gal, ngal, c0, nrow, i, ui, vi, wi, wn, inv_lambda, spec, sign,
                                   res);
    for (; c0 < nch; c0++)
        add_sources_block<PREC, 1>(gal, ngal, c0, nrow, i, ui, vi, wi, wn, inv_lambda, spec, sign,
                                   res);
}

void launch_add_sources(hipStream_t s, int prec, unsigned nch, unsigned long nrow,
                        const double *u, const double *v, const double *w, const double *wn,
                        const double *inv_lambda, const double *spec, const GalaxyGeom *gal,
                        unsigned ngal, double sign, void *res)
{
    dim3 grid((unsigned)((nrow + 255) / 256));
    if (prec == 0)
        add_sources_kernel<0><<<grid, 256, 0, s>>>(nch, nrow, u, v, w, wn, inv_lambda, spec, gal,
                                                    ngal, sign, res);
    else
        add_sources_kernel<1><<<grid, 256, 0, s>>>(nch, nrow, u, v, w, wn, inv_lambda, spec, gal,
                                                    ngal, sign, res);
}

template <int PREC>
__global__ void add_noise_kernel(unsigned long nvis, double sigma, uint64_t seed, void *res)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nvis) return;
    // Philox4x32-10 (rl2_math.h) of counter (i, 0x5eed, 0) under the seed -> Box-Muller
    const uint32_t ctr[4] = {(uint32_t)i, (uint32_t)(i >> 32), 0x5eedu, 0u};
    const uint32_t key[2] = {(uint32_t)seed, (uint32_t)(seed >> 32)};
    uint32_t rr[4];
    philox4x32_10(ctr, key, rr);
    const uint4 r = make_uint4(rr[0], rr[1], rr[2], rr[3]);
    // 53-bit uniforms in (0, 1]
    double u1 = ((double)(((uint64_t)r.x << 21) ^ (r.y >> 11)) + 1.0) * (1.0 / 9007199254740992.0);
    double u2 = ((double)(((uint64_t)r.z << 21) ^ (r.w >> 11)) + 0.5) * (1.0 / 9007199254740992.0);
    double rad = sqrt(-2.0 * log(u1));
    double sn, cs;
    sincospi(2.0 * u2, &sn, &cs);
    double2 x = load_res(res, PREC, i);
    x.x += sigma * rad * cs;
    x.y += sigma * rad * sn;
    store_res(res, PREC, i, x);
}

void launch_add_noise(hipStream_t s, int prec, unsigned long nvis, double sigma, uint64_t seed,
                      void *res)
{
    dim3 grid((unsigned)((nvis + 255) / 256));
    if (prec == 0)
        add_noise_kernel<0><<<grid, 256, 0, s>>>(nvis, sigma, seed, res);
    else
        add_noise_kernel<1><<<grid, 256, 0, s>>>(nvis, sigma, seed, res);
}

// ------------------------------------------------------------------ extraction + gridding
// Deterministic accumulation.  The gridded sums of a cell are kept as integers, so the
// order in which work-groups and threads add them does not change a single bit:
//  - a value x (a visibility component, or sigma^2) is carried as rint(x * 2^S), with S
//    chosen per launch from a bound B >= |x| (the residual's bound plus the galaxy's flux;
//    the largest sigma^2) so that B * 2^S * (rows of a work-group) <= 2^62;
//  - a work-group adds its runs in LDS as int64 (the slot sums of a channel cover at most
//    the work-group's rows, so they stay below 2^62);
//  - the flush splits each slot sum into its high word (arithmetic shift by 32) and its low
//    32 bits, added by integer atomics into two 64-bit accumulators per cell and component
//    (no carries are lost: the low sums stay below 2^64 for fewer than 2^32 flushes);
//  - compaction recombines hi * 2^32 + lo and scales by 2^-S.
// Each visibility is rounded on its own (runs of a cell are then added as integers), and
// every gridding path takes S from one bound (the most terms any of them puts in a slot
// between flushes), so the facet is the same bit for bit whatever the variant, the batch
// path, the order of work-groups or the run.  A term's rounding is at most 2^-(S+1), below
// B * 2^-48 for 16 channels, and the sum itself is exact, so the facet agrees with the
// reference's sequential FP64 sums to their own rounding.
// Accumulator layout: 7 arrays of facet^2 words: re hi, re lo, im hi, im lo, sigma^2 hi,
// sigma^2 lo (uint64, two's complement), weight (double, integer-valued).
enum { kAccReHi = 0, kAccReLo, kAccImHi, kAccImLo, kAccS2Hi, kAccS2Lo, kAccW, kAccWords };

__device__ inline long long fx_round(double x, double scale)
{
    return (long long)rint(x * scale);
}

__device__ inline void fx_flush(unsigned long long *hi, unsigned long long *lo, long long v)
{
    atomicAdd(hi, (unsigned long long)(v >> 32));
    atomicAdd(lo, (unsigned long long)(v & 0xffffffffll));
}

// Variants 2-4.  Each thread owns RPT consecutive sorted rows and, per channel, adds runs
// of consecutive visibilities that fall in the same cell in registers before one LDS
// update per run: in the dense uv core, where many rows share a cell, this removes most of
// the same-address LDS atomics that serialise across a wave.  A channel inserts at most
// RPT*256 runs into the HS-slot table (HS >= RPT*256, so probing always finds a slot);
// flush as variant 0.
// SUB: first apply the previous galaxy's post-fit update (a.sfit, a.srnd) to each of the
// thread's visibilities and write it back, then grid the updated value: the subtraction and
// the next extraction share one pass over the residual, and every visibility gets the same
// arithmetic, in the same order, as subtract_kernel followed by this kernel.
// LAZY: the table keeps its cells from one channel to the next and is flushed only when
// another channel's runs might not fit (more than HS - RPT*256 slots in use) and after the
// last channel.  Neighbouring channels put a dense-core visibility in the same cell, so the
// global atomics of a cell are made once for several channels; the integer sums make the
// facet the same bit for bit whenever the flushes happen.
template <int MODE, int PREC, int RPT, int HS, bool SUB = false, bool LAZY = false>
__global__ __launch_bounds__(256) void grid_run_kernel(GridLaunch a)
{
    constexpr int BS = 256;
    static_assert(HS >= RPT * BS, "a free slot must exist for every run of a channel");
    constexpr int HBITS = (HS == 2048) ? 11 : (HS == 1024) ? 10 : (HS == 4096) ? 12 : 9;
    static_assert((1 << HBITS) == HS, "hash size must be a power of two");
    static_assert(RPT * BS <= 4096, "slot sums of a channel must stay below 2^62");
    __shared__ uint32_t hkey[HS];
    __shared__ unsigned long long hre[HS], him[HS], hs2[HS];  // rint(x * 2^S), int64
    __shared__ uint32_t hcnt[HS];
    __shared__ uint32_t hlist[HS];
    __shared__ uint32_t hn;
    const int tid = threadIdx.x;
    for (int s = tid; s < HS; s += BS) {
        hkey[s] = kEmpty;
        hre[s] = 0ull;
        him[s] = 0ull;
        hs2[s] = 0ull;
        hcnt[s] = 0;
    }
    if (tid == 0) hn = 0;
    const unsigned long row0 = (unsigned long)blockIdx.x * (RPT * BS) + (unsigned long)tid * RPT;
    const unsigned long ncell = (unsigned long)a.facet * a.facet;
    const double inv_inc = 1.0 / a.inc;
    unsigned long long *acc = (unsigned long long *)a.acc;
    double *acc_w = a.acc + kAccW * ncell;
    // a run's sums are already integers (each visibility rounded on its own, so the run
    // length, and with it the variant, does not change a bit)
    auto emit = [&](uint32_t key, long long xr, long long xi, long long xs, uint32_t n) {
        uint32_t h = (key * 2654435761u) >> (32 - HBITS);
        while (true) {
            const uint32_t prev = atomicCAS(&hkey[h], kEmpty, key);
            if (prev == kEmpty) hlist[atomicAdd(&hn, 1u)] = h;
            if (prev == kEmpty || prev == key) break;
            h = (h + 1) & (HS - 1);
        }
        if (MODE != 2) {
            atomicAdd(&hre[h], (unsigned long long)xr);
            atomicAdd(&him[h], (unsigned long long)xi);
        }
        atomicAdd(&hs2[h], (unsigned long long)xs);
        atomicAdd(&hcnt[h], n);
    };
    // the rows' u, v and phase numerator p = ul + vm + wn stay in registers for all
    // channels (the channel only scales them)
    double ru[RPT], rv[RPT], rp[RPT], rps[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        const unsigned long i = row0 + k;
        const bool in = i < a.nrow;
        ru[k] = in ? a.u[i] : 0.;
        rv[k] = in ? a.v[i] : 0.;
        const double wi = (in && MODE == 0) ? a.w[i] : 0.;
        rp[k] = (in && MODE == 0) ? ru[k] * a.g.l0 + rv[k] * a.g.m0 + wi * a.g.n0 : 0.;
        rps[k] = (in && SUB) ? ru[k] * a.sfit.l0 + rv[k] * a.sfit.m0 + wi * a.sfit.n0 : 0.;
    }
    __syncthreads();
    for (unsigned c = 0; c < a.nch; c++) {
        const double wn = a.wn[c], inv_lambda = a.inv_lambda[c];
        const double wn2 = wn * wn, spectra = a.spec[c];
        uint32_t rkey = kEmpty, rn = 0;
        long long rre = 0, rim = 0, rs2 = 0;
        // the thread's RPT consecutive visibilities are loaded together, so each load
        // instruction's cache lines are still resident for the next one (issued one row
        // at a time between the gridding work, they were fetched from HBM ~3 times over)
        float vs2[RPT];
        double2 vres[RPT];
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            const unsigned long i = row0 + k;
            const size_t idx = (size_t)c * a.nrow + i;
            vs2[k] = i < a.nrow ? a.s2f[idx] : -1.f;
            vres[k] = (MODE != 2 && i < a.nrow) ? load_res(a.res, PREC, idx) : make_double2(0., 0.);
        }
        if (SUB) {
#pragma unroll
            for (int k = 0; k < RPT; k++) {
                const unsigned long i = row0 + k;
                if (i >= a.nrow) continue;
                const size_t idx = (size_t)c * a.nrow + i;
                const double2 r = subtract_vis(a.sfit, a.srnd, rps[k], ru[k], rv[k], wn2,
                                               spectra, inv_lambda, vres[k]);
                store_res(a.res_w, PREC, idx, r);
                // the value a separate pass would read back
                vres[k] = PREC == 0 ? r : make_double2((double)(float)r.x, (double)(float)r.y);
            }
        }
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            const unsigned long i = row0 + k;
            if (i >= a.nrow) continue;
            const float s2 = vs2[k];
            if (signbit(s2)) continue;  // flagged
            const double u = ru[k], v = rv[k];
            uint32_t key;
            if (!cell_index_fast(u, v, inv_lambda, a.len, a.inc, inv_inc, a.facet, &key)) continue;
            double xr = 0., xi = 0.;
            if (MODE == 0) {
                // visGal = round model + (visData - visSkyMod), then shift by -k(ul+vm+wn)
                // (source_extraction.c:51-65); the phase k p in revolutions is p / lambda.
                const double p = rp[k];
                const double shape = model_shape_rsq(a.g, u, v, wn2, spectra);
                double sn, cs;
                sincos_rev64(p * inv_lambda, sn, cs);
                const double2 r = vres[k];
                const double gre = shape * cs + r.x;
                const double gim = shape * sn + r.y;
                xr = gre * cs - gim * (-sn);
                xi = gre * (-sn) + gim * cs;
            } else if (MODE == 1) {
                const double2 r = vres[k];
                xr = r.x;
                xi = r.y;
            }
            const long long ir = MODE != 2 ? fx_round(xr, a.fx_scale) : 0;
            const long long ii = MODE != 2 ? fx_round(xi, a.fx_scale) : 0;
            const long long is = fx_round((double)s2, a.fs_scale);
            if (key == rkey) {
                rre += ir;
                rim += ii;
                rs2 += is;
                rn++;
            } else {
                if (rn) emit(rkey, rre, rim, rs2, rn);
                rkey = key;
                rre = ir;
                rim = ii;
                rs2 = is;
                rn = 1;
            }
        }
        if (rn) emit(rkey, rre, rim, rs2, rn);
        __syncthreads();
        const uint32_t nocc = hn;
        if (LAZY && c + 1 < a.nch && nocc <= (uint32_t)(HS - RPT * BS)) continue;
        for (uint32_t j = tid; j < nocc; j += BS) {
            const uint32_t s = hlist[j];
            const uint32_t key = hkey[s];
            if (MODE != 2) {
                fx_flush(acc + kAccReHi * ncell + key, acc + kAccReLo * ncell + key,
                         (long long)hre[s]);
                fx_flush(acc + kAccImHi * ncell + key, acc + kAccImLo * ncell + key,
                         (long long)him[s]);
            }
            fx_flush(acc + kAccS2Hi * ncell + key, acc + kAccS2Lo * ncell + key,
                     (long long)hs2[s]);
            unsafeAtomicAdd(&acc_w[key], (double)hcnt[s]);  // integer-valued: exact
            hkey[s] = kEmpty;
            hre[s] = 0ull;
            him[s] = 0ull;
            hs2[s] = 0ull;
            hcnt[s] = 0;
        }
        __syncthreads();
        if (tid == 0) hn = 0;
        __syncthreads();
    }
}

// ---- extraction's default: one LDS table per work-group with several copies of every sum
// Sorted rows put a wave's visibilities of a channel into two to four cells (64 rows of a
// 197-dish observation into 1.7 cells at 296 columns, 3.2 at 924), so a table with one sum per
// cell made the LDS atomics of 64 lanes wait for each other on one address: they were half of
// the extraction.  Here lane l adds to copy l % 4 of a cell's sums, which are in different
// banks, and the copies are added when the table is flushed.  256 threads of 2 rows and 256
// cells of 4 copies: 30 KB, five work-groups per CU, the 20 waves that 100 registers allow (with
// the subtraction 16); 512 rows and all channels of that array have 20 to 120 cells.
// 148M visibilities (complex128, 16 channels) take 0.78 ms into 296 columns and 1.05 into 924
// (runs merged in registers, one sum per cell: 1.42), 1.27 with the subtraction (1.62), 29M in
// complex64 0.23 ms (0.37), 3.9M in 4 channels 27 us (51).  The bytes take 0.61 ms (1.09 with
// the subtraction) at the rate of a large copy; what is left is FP64 arithmetic (over half of
// the issue slots) and the LDS atomics.  512 threads and 512 cells take 0.92, 1.13, 1.32 and
// 0.27 ms (16 waves, and a work-group's sparse rows keep more waves waiting), 128 threads 25%
// more on the smallest, 128 cells 1% to 4%, 2 copies 4%, a row per thread 25%; runs kept in
// registers across channels 9%; loading a channel ahead gives nothing.
// A visibility that finds no place in kCellProbes steps goes to the accumulators directly, so
// the table has no size that must suffice, and it is flushed when three quarters are in use
// (looked at every four channels) and at the end.  The integer sums make the facet the same
// bit for bit however the visibilities are spread over copies and flushes.
// Values are rounded by adding 1.5 * 2^52 (|x| 2^S < 2^51 by fx_scales, which needs finite
// bounds: the host takes the kernel above otherwise); a NaN counts as 0, as its conversion did.
constexpr int kCellBS = 256, kCellRows = 2, kCellSlots = 256, kCellCopies = 4, kCellProbes = 8;
struct CellTable {
    unsigned long long sum[3][kCellSlots * kCellCopies];  // re, im, sigma^2
    uint32_t cnt[kCellSlots * kCellCopies];
    uint32_t key[kCellSlots], list[kCellSlots];
    uint32_t used;
};

__device__ inline long long fx_round51(double x, double scale)
{
    constexpr double kRound = 6755399441055744.;
    return (long long)(__builtin_bit_cast(uint64_t, fma(x, scale, kRound)) -
                       __builtin_bit_cast(uint64_t, kRound));
}

__device__ inline void cell_clear(CellTable &T)
{
    for (int k = threadIdx.x; k < kCellSlots * kCellCopies; k += kCellBS) {
        T.sum[0][k] = T.sum[1][k] = T.sum[2][k] = 0ull;
        T.cnt[k] = 0;
    }
    static_assert(kCellSlots <= kCellBS, "a key per thread");
    if (threadIdx.x < kCellSlots) T.key[threadIdx.x] = kEmpty;
    if (threadIdx.x == 0) T.used = 0;
}

__device__ inline void cell_add(CellTable &T, double *accd, unsigned long ncell, uint32_t key,
                                long long re, long long im, long long s2, uint32_t n)
{
    uint32_t h = (key * 2654435761u) >> 24;
    static_assert(kCellSlots == 1 << 8, "hash bits");
#pragma unroll 1
    for (int p = 0; p < kCellProbes; p++) {
        uint32_t k = __hip_atomic_load(&T.key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k == kEmpty) {
            k = atomicCAS(&T.key[h], kEmpty, key);
            if (k == kEmpty) {
                T.list[atomicAdd(&T.used, 1u)] = h;
                k = key;
            }
        }
        if (k == key) {
            const uint32_t at = h * kCellCopies + (threadIdx.x & (kCellCopies - 1));
            atomicAdd(&T.sum[0][at], (unsigned long long)re);
            atomicAdd(&T.sum[1][at], (unsigned long long)im);
            atomicAdd(&T.sum[2][at], (unsigned long long)s2);
            atomicAdd(&T.cnt[at], n);
            return;
        }
        h = (h + 1) & (kCellSlots - 1);
    }
    unsigned long long *acc = (unsigned long long *)accd;
    fx_flush(acc + kAccReHi * ncell + key, acc + kAccReLo * ncell + key, re);
    fx_flush(acc + kAccImHi * ncell + key, acc + kAccImLo * ncell + key, im);
    fx_flush(acc + kAccS2Hi * ncell + key, acc + kAccS2Lo * ncell + key, s2);
    unsafeAtomicAdd(&accd[kAccW * ncell + key], (double)n);
}

// The table's sums to the accumulators, and the table empty again; by the whole work-group,
// with a barrier before it and the last one inside.
__device__ inline void cell_flush(CellTable &T, double *accd, unsigned long ncell)
{
    const uint32_t nocc = T.used;
    unsigned long long *acc = (unsigned long long *)accd;
    for (uint32_t j = threadIdx.x; j < nocc * 4; j += kCellBS) {
        const uint32_t s = T.list[j >> 2], q = j & 3, key = T.key[s];
        unsigned long long t = 0;
#pragma unroll
        for (uint32_t i = 0; i < kCellCopies; i++) {  // starting at another bank for each cell
            const uint32_t at = s * kCellCopies + ((i + s) & (kCellCopies - 1));
            if (q < 3) {
                t += T.sum[q][at];
                T.sum[q][at] = 0ull;
            } else {
                t += T.cnt[at];
                T.cnt[at] = 0;
            }
        }
        if (q < 3)
            fx_flush(acc + (2 * q) * ncell + key, acc + (2 * q + 1) * ncell + key, (long long)t);
        else
            unsafeAtomicAdd(&accd[kAccW * ncell + key], (double)t);  // integer-valued: exact
    }
    static_assert(kAccReHi == 0 && kAccImHi == 2 && kAccS2Hi == 4, "accumulator order");
    __syncthreads();
    for (uint32_t j = threadIdx.x; j < nocc; j += kCellBS) T.key[T.list[j]] = kEmpty;
    if (threadIdx.x == 0) T.used = 0;
    __syncthreads();
}

// One visibility of a galaxy's facet: the round model added, shifted to the galaxy
// (source_extraction.c:51-65), as integers of the facet's scale, with its cell; false when it is
// flagged or outside.
struct CellTerm {
    uint32_t key;
    long long re, im, s2;
};
template <class Exact>
__device__ inline bool cell_term(CellTerm &o, const GridLaunch &a, double u_inc, double v_inc,
                                 double mid, double kk, double p, double2 r, float s2, double wn2,
                                 double spectra, double inv_lambda, const Exact &exact)
{
    if (signbit(s2)) return false;
    if (!cell_index_scaled(u_inc, v_inc, inv_lambda, mid, a.len, a.inc, a.facet, exact, &o.key))
        return false;
    const double shape = model_shape_kk(a.g, kk, wn2, spectra);
    double sn, cs;
    sincos_rev64(p * inv_lambda, sn, cs);  // the phase k p in revolutions is p / lambda
    const double gre = shape * cs + r.x;
    const double gim = shape * sn + r.y;
    const double xr = gre * cs - gim * (-sn);
    const double xi = gre * (-sn) + gim * cs;
    const bool nan = __builtin_isunordered(xr, xi);
    o.re = nan ? 0 : fx_round51(xr, a.fx_scale);
    o.im = nan ? 0 : fx_round51(xi, a.fx_scale);
    o.s2 = fx_round51((double)s2, a.fs_scale);  // never a NaN (pack_sigma_kernel)
    return true;
}

// SUB: the previous galaxy's post-fit update in the same pass, as grid_run_kernel.
// Each work-group takes its rows' channels from blockIdx.y * channels on.
template <int PREC, bool SUB>
__global__ __launch_bounds__(kCellBS, SUB ? 4 : 5) void grid_cell_kernel(GridLaunch a,
                                                                         unsigned channels)
{
    constexpr int RPT = kCellRows;
    static_assert(RPT == 2, "a pair of rows");
    __shared__ CellTable T;
    cell_clear(T);
    // The work-groups of the sorted order's two ends first: its sparse corners, whose rows have
    // cells of their own, take two to four times as long as the others and would otherwise run
    // alone at the end (115 us of 270 on 29M visibilities).
    const unsigned block =
        blockIdx.x & 1 ? gridDim.x - 1 - blockIdx.x / 2 : blockIdx.x / 2;
    const unsigned long row0 =
        (unsigned long)block * (RPT * kCellBS) + (unsigned long)threadIdx.x * RPT;
    const unsigned long ncell = (unsigned long)a.facet * a.facet;
    const double inv_inc = 1.0 / a.inc, mid = a.len * inv_inc;
    // What a row keeps for all channels; its u and v in metres only for the rare exact cell
    // index, so they are read again there.  A row past the end reads the last one's values and
    // counts as flagged.
    double ru[RPT], rv[RPT], rp[RPT], rps[RPT], rk[RPT], rkf[RPT];
    bool ok[RPT];
    using Res = typename std::conditional<PREC == 0, double2, float2>::type;
    const Res *pr[RPT];
    const float *ps[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        ok[k] = row0 + k < a.nrow;
        const unsigned long i = ok[k] ? row0 + k : a.nrow - 1;
        const double u = a.u[i], v = a.v[i], w = a.w[i];
        ru[k] = u * inv_inc;
        rv[k] = v * inv_inc;
        rp[k] = u * a.g.l0 + v * a.g.m0 + w * a.g.n0;
        rk[k] = model_kk(a.g, u, v);  // SUB: that of srnd too (the host checks e = 0 in both)
        rps[k] = SUB ? u * a.sfit.l0 + v * a.sfit.m0 + w * a.sfit.n0 : 0.;
        rkf[k] = SUB ? model_kk(a.sfit, u, v) : 0.;
        pr[k] = (const Res *)a.res + i;
        ps[k] = a.s2f + i;
    }
    __syncthreads();
    const unsigned c0 = blockIdx.y * channels, c1 = min(a.nch, c0 + channels);
    for (unsigned c = c0; c < c1; c++) {
        const double wn = a.wn[c], inv_lambda = a.inv_lambda[c];
        const double wn2 = wn * wn, spectra = a.spec[c];
        // both rows' values together: each line is still there for the second load
        float vs2[RPT];
        double2 vres[RPT];
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            const Res r = pr[k][(size_t)c * a.nrow];
            const float s2 = ps[k][(size_t)c * a.nrow];
            vres[k] = make_double2((double)r.x, (double)r.y);
            vs2[k] = ok[k] ? s2 : -1.f;
        }
        if (SUB) {
#pragma unroll
            for (int k = 0; k < RPT; k++) {
                const double2 r = subtract_vis_kk(a.sfit, a.srnd, rps[k], rkf[k], rk[k], wn2,
                                                  spectra, inv_lambda, vres[k]);
                if (ok[k]) store_res(a.res_w, PREC, (size_t)c * a.nrow + row0 + k, r);
                // the value a separate pass would read back
                vres[k] = PREC == 0 ? r : make_double2((double)(float)r.x, (double)(float)r.y);
            }
        }
        CellTerm t[RPT];
        bool in[RPT];
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            in[k] = cell_term(t[k], a, ru[k], rv[k], mid, rk[k], rp[k], vres[k], vs2[k], wn2,
                              spectra, inv_lambda, [&](double *u, double *v) {
                                  const unsigned long i = row0 + k;  // not flagged: a row
                                  *u = a.u[i];
                                  *v = a.v[i];
                              });
        }
        const bool pair = in[0] && in[1] && t[0].key == t[1].key;
        if (pair) {
            t[0].re += t[1].re;
            t[0].im += t[1].im;
            t[0].s2 += t[1].s2;
        }
        // one call site: a lane's second visibility in another cell takes another turn
        bool more = in[0] || in[1];
        bool first = in[0];
        while (more) {
            const uint32_t key = first ? t[0].key : t[1].key;
            const long long re = first ? t[0].re : t[1].re, im = first ? t[0].im : t[1].im,
                            s2 = first ? t[0].s2 : t[1].s2;
            cell_add(T, a.acc, ncell, key, re, im, s2, first && pair ? 2u : 1u);
            more = first && in[1] && !pair;
            first = false;
        }
        if ((c & 3) == 3 && c + 1 < c1) {
            __syncthreads();
            const uint32_t used = T.used;
            __syncthreads();  // every thread has read it before any adds a cell
            if (used > kCellSlots * 3 / 4) cell_flush(T, a.acc, ncell);
        }
    }
    __syncthreads();
    cell_flush(T, a.acc, ncell);
}

template <int MODE, int PREC>
static void launch_grid_variant(hipStream_t s, const GridLaunch &a)
{
    if (MODE == 0 && tuning().grid_variant == 5 && a.finite &&
        !(a.sub && (a.g.e1 != 0. || a.g.e2 != 0. || a.srnd.e1 != 0. || a.srnd.e2 != 0.))) {
        // A work-group goes through its channels one after the other, 3 to 5 us each, and with many
        // of them its rows' cells outgrow the table (a cell moves with the wavelength).  So the
        // channels are shared out: 16 at most to a work-group, and with few rows fewer, four at
        // least, until the work-groups fill the chip twice (one wave of them ends with its
        // slowest).  Merging runs / all channels in one work-group / shared out: 2,760 rows of 64
        // channels into 134 columns 233 / 343 / 45 us, 20,160 of 256 into 142 columns 766 / 1,288 /
        // 110, 201,600 of 64 into 82 columns 246 / 337 / 121, 714,000 of 128 into 1,110 columns
        // 2.66 / 2.51 / 2.03 ms, 685,440 of 128 into 1,216 columns 3.39 / 3.61 / 2.80 ms.  Eight
        // channels at most are 0 to 5% slower near the array's core and as much faster far from
        // it; 32 up to 20% slower.
        constexpr unsigned rows = kCellRows * kCellBS;
        const unsigned blocks = (unsigned)((a.nrow + rows - 1) / rows);
        const unsigned fill = 2 * (a.sub ? 4 : 5) * num_cus();
        const unsigned shares =  // (65,535 at most: the launch's limit)
            std::min(65535u, std::max({1u, fill / blocks, (a.nch + 15) / 16}));
        const unsigned channels = ((a.nch + shares - 1) / shares + 3) / 4 * 4;
        const dim3 grid(blocks, (a.nch + channels - 1) / channels);
        if (a.sub)
            grid_cell_kernel<PREC, true><<<grid, kCellBS, 0, s>>>(a, channels);
        else
            grid_cell_kernel<PREC, false><<<grid, kCellBS, 0, s>>>(a, channels);
        return;
    }
    if (tuning().grid_variant == 5) {
        // runs of 2 rows, 1024 slots, flushed when another channel might not fit
        constexpr int RPT = 2;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        if (MODE == 0 && a.sub)
            grid_run_kernel<MODE, PREC, RPT, 1024, true, true><<<grid, 256, 0, s>>>(a);
        else
            grid_run_kernel<MODE, PREC, RPT, 1024, false, true><<<grid, 256, 0, s>>>(a);
    } else if (tuning().grid_variant == 6) {
        // runs of 4 rows, 2048 slots, flushed when another channel might not fit
        constexpr int RPT = 4;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        if (MODE == 0 && a.sub)
            grid_run_kernel<MODE, PREC, RPT, 2048, true, true><<<grid, 256, 0, s>>>(a);
        else
            grid_run_kernel<MODE, PREC, RPT, 2048, false, true><<<grid, 256, 0, s>>>(a);
    } else if (tuning().grid_variant == 2) {
        constexpr int RPT = 8;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        grid_run_kernel<MODE, PREC, RPT, 2048><<<grid, 256, 0, s>>>(a);
    } else if (tuning().grid_variant == 3) {
        constexpr int RPT = 4;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        if (MODE == 0 && a.sub)
            grid_run_kernel<MODE, PREC, RPT, 1024, true><<<grid, 256, 0, s>>>(a);
        else
            grid_run_kernel<MODE, PREC, RPT, 1024><<<grid, 256, 0, s>>>(a);
    } else if (tuning().grid_variant == 4) {
        constexpr int RPT = 4;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        grid_run_kernel<MODE, PREC, RPT, 2048><<<grid, 256, 0, s>>>(a);
    } else if (tuning().grid_variant == 1) {
        constexpr int RPT = 2;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        grid_run_kernel<MODE, PREC, RPT, 1024><<<grid, 256, 0, s>>>(a);
    } else {
        // runs of 2 rows: 512 rows per work-group and a 512-slot table (18 KB of LDS)
        constexpr int RPT = 2;
        dim3 grid((unsigned)((a.nrow + RPT * 256 - 1) / (RPT * 256)));
        grid_run_kernel<MODE, PREC, RPT, 512><<<grid, 256, 0, s>>>(a);
    }
}

void launch_grid(hipStream_t s, const GridLaunch &a)
{
    if (a.mode == 0) {
        if (a.prec == 0)
            launch_grid_variant<0, 0>(s, a);
        else
            launch_grid_variant<0, 1>(s, a);
    } else if (a.mode == 1) {
        launch_grid_variant<1, 0>(s, a);
    } else {
        launch_grid_variant<2, 0>(s, a);
    }
}

// ------------------------------------------------------------------ compaction
// Cells with weight != 0 in row-major order (evaluate_uv_grid.c:196-210 and :113-133):
//   vis = sum_vis * w / sum_sigma2, sigma2 = sum_sigma2 / w^2, (u,v) = cell centre.
// Two launches: the cells of every tile are counted, then a work-group per tile adds the counts
// of the tiles before it (at most a few hundred words from L2, instead of a scan of its own)
// and writes its cells with every copy of them that the likelihood reads.  Bound by the latency
// of its loads: consecutive lanes take consecutive cells, kCompactPT loads in flight each.
// An extracted facet of 1,024 grid cells takes 4 + 6 us (a count, a scan, a write of 16 cells
// in a row per thread and a copying launch: 5 + 4 + 20 + 5 us), of 60,000 cells 5 + 13 (6 + 5 +
// 61 + 6).
constexpr int kCompactBS = 256, kCompactPT = 4, kCompactTile = kCompactBS * kCompactPT;
constexpr int kCompactW = kCompactBS / 64;

__host__ __device__ inline unsigned compact_tiles(unsigned long ncell)
{
    return (unsigned)((ncell + kCompactTile - 1) / kCompactTile);
}

size_t compact_scratch_words(unsigned facet)
{
    return compact_tiles((unsigned long)facet * facet) + 1;
}

__device__ inline void compact_count_tile(unsigned blk, const double *acc_w, unsigned long ncell,
                                          unsigned *bcount)
{
    __shared__ unsigned part[kCompactW];
    const unsigned long base = (unsigned long)blk * kCompactTile + threadIdx.x;
    unsigned cnt = 0;
#pragma unroll
    for (int k = 0; k < kCompactPT; k++) {
        const unsigned long p = base + k * kCompactBS;
        cnt += (unsigned)__popcll(__ballot(p < ncell && acc_w[p < ncell ? p : 0] != 0.));
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned t = 0;
        for (int i = 0; i < kCompactW; i++) t += part[i];
        bcount[blk] = t;
    }
}

__global__ __launch_bounds__(kCompactBS) void compact_count_kernel(const double *acc_w,
                                                                   unsigned long ncell,
                                                                   unsigned *bcount)
{
    compact_count_tile(blockIdx.x, acc_w, ncell, bcount);
}

// Accumulators of cell p: FX (device gridding) the integer layout above, scaled back by
// 2^-S; otherwise four double arrays (re, im, sigma^2, weight) given by a caller.
template <bool FX>
__device__ inline void acc_read(double *acc, unsigned long ncell, unsigned long p,
                                double fx_unscale, double fs_unscale, double &re, double &im,
                                double &sg)
{
    if (FX) {
        const unsigned long long *q = (const unsigned long long *)acc;
        auto get = [&](int hi, int lo, double unscale) {
            const unsigned long long l = q[lo * ncell + p];
            const long long h = (long long)q[hi * ncell + p] + (long long)(l >> 32);
            return ((double)h * 4294967296.0 + (double)(l & 0xffffffffull)) * unscale;
        };
        re = get(kAccReHi, kAccReLo, fx_unscale);
        im = get(kAccImHi, kAccImLo, fx_unscale);
        sg = get(kAccS2Hi, kAccS2Lo, fs_unscale);
    } else {
        re = acc[p];
        im = acc[ncell + p];
        sg = acc[2 * ncell + p];
    }
}

template <bool FX>
__device__ inline void acc_clear(double *acc, unsigned long ncell, unsigned long p)
{
    if (FX) {
        unsigned long long *q = (unsigned long long *)acc;
        for (int k = 0; k < kAccW; k++) q[k * ncell + p] = 0ull;
        acc[kAccW * ncell + p] = 0.;
    } else {
        for (int k = 0; k < 4; k++) acc[k * ncell + p] = 0.;
    }
}

// Cell i's packed data and record offsets for the fused Newton passes (cell n: the zero pad
// cell); offsets only for grid facets with records (facet <= kRecFacet).
__device__ inline void pack_cell_records(unsigned i, double re, double im, const uint32_t *cid,
                                         uint32_t c, unsigned facet, double2 *dc, uint32_t *loff)
{
    dc[i] = make_double2(re, im);
    if (cid && facet <= kRecFacet)
        loff[i] = ((c >> 16) * kRecBytes) << 16 | (c & 0xffffu) * kRecBytes;
}

// One work-group's tile of the compaction (tile `blk` of the nb tiles of one facet).
template <bool FX>
__device__ inline void compact_write_tile(unsigned blk, unsigned nb, double *acc, unsigned facet,
                                          unsigned long ncell, double len, const unsigned *bcount,
                                          const CompactOut &C, double fx_unscale,
                                          double fs_unscale)
{
    __shared__ unsigned part[kCompactW], count[kCompactPT][kCompactW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double *acc_w = acc + (FX ? kAccW : 3) * ncell;
    const unsigned long base = (unsigned long)blk * kCompactTile + threadIdx.x;
    double wgt[kCompactPT];
#pragma unroll
    for (int k = 0; k < kCompactPT; k++) {
        const unsigned long p = base + k * kCompactBS;
        wgt[k] = p < ncell ? acc_w[p] : 0.;
    }
    unsigned before = 0;
    for (unsigned t = threadIdx.x; t < blk; t += kCompactBS) before += bcount[t];
    for (int off = 32; off >= 1; off >>= 1) before += __shfl_xor(before, off);
    if (lane == 0) part[wave] = before;
    unsigned rank[kCompactPT];
#pragma unroll
    for (int k = 0; k < kCompactPT; k++) {
        const unsigned long long mask = __ballot(wgt[k] != 0.);
        rank[k] = (unsigned)__popcll(mask & ((1ull << lane) - 1ull));
        if (lane == 0) count[k][wave] = (unsigned)__popcll(mask);
    }
    __syncthreads();
    unsigned n = 0;
#pragma unroll
    for (int w = 0; w < kCompactW; w++) n += part[w];
    const double inc = 2 * len / facet;
    if (C.ctr) {  // centre of grid index k, the same expression as uu / vv below
        const unsigned k = blk * kCompactBS + threadIdx.x;
        if (k < facet) C.ctr[k] = (k + 0.5) * inc - len;
    }
#pragma unroll
    for (int k = 0; k < kCompactPT; k++) {
        const unsigned long p = base + k * kCompactBS;
        unsigned at = n + rank[k];
#pragma unroll
        for (int w = 0; w < kCompactW; w++) {
            const unsigned c = count[k][w];
            at += w < wave ? c : 0;
            n += c;
        }
        if (C.sum_w && p < ncell) C.sum_w[p] = wgt[k];
        if (wgt[k] == 0.) continue;
        double re, im, sg;
        acc_read<FX>(acc, ncell, p, fx_unscale, fs_unscale, re, im, sg);
        const double dre = re * wgt[k] / sg, dim = im * wgt[k] / sg;
        const double s2 = sg / (wgt[k] * wgt[k]);
        const unsigned q = (unsigned)p, j = q / facet, i = q - j * facet;
        const double u = (i + 0.5) * inc - len, v = (j + 0.5) * inc - len;
        const uint32_t id = (j << 16) | i;
        C.dre[at] = dre;
        C.dim[at] = dim;
        C.s2[at] = s2;
        C.uu[at] = u;
        C.vv[at] = v;
        if (C.cid) C.cid[at] = id;
        if (C.pk) {
            const double w = 1.0 / s2;
            C.pk[at] = make_float4((float)u, (float)v, (float)dre, (float)dim);
            C.invs2[at] = (float)w;
            C.invs2_64[at] = w;
            pack_cell_records(at, dre, dim, C.cid, id, facet, C.dc, C.loff);
        }
        if (C.h_vis) {
            C.h_vis[at] = make_double2(dre, dim);
            C.h_s2[at] = s2;
            C.h_uu[at] = u;
            C.h_vv[at] = v;
        }
        acc_clear<FX>(acc, ncell, p);
    }
    if (blk == nb - 1 && threadIdx.x == 0) {
        *C.n_out = n;
        if (C.n_host) *C.n_host = n;
        // zero pad cell after the last one (the arrays hold facet^2 + 1 entries): lanes past
        // the end of a chunk read it instead of masking their data
        if (C.cid) {
            C.dre[n] = 0.;
            C.dim[n] = 0.;
            C.cid[n] = 0;
        }
        if (C.pk) {
            C.invs2_64[n] = 0.;
            pack_cell_records(n, 0., 0., C.cid, 0u, facet, C.dc, C.loff);
        }
    }
}

template <bool FX>
__global__ __launch_bounds__(kCompactBS) void compact_write_kernel(double *acc, unsigned facet,
                                                                   unsigned long ncell, double len,
                                                                   const unsigned *bcount,
                                                                   CompactOut C, double fx_unscale,
                                                                   double fs_unscale)
{
    compact_write_tile<FX>(blockIdx.x, gridDim.x, acc, facet, ncell, len, bcount, C, fx_unscale,
                           fs_unscale);
}

// ---- batched compaction: grid.y = target of a BatchDesc; targets beyond desc->ntarget and
// blocks beyond a target's facet exit at once, so one launch shape serves every batch.
__global__ __launch_bounds__(kCompactBS) void compact_count_batch_kernel(const BatchDesc *desc)
{
    const unsigned t = blockIdx.y;
    if (t >= desc->ntarget) return;
    const BatchCompact &C = desc->compact[t];
    const unsigned long ncell = (unsigned long)C.facet * C.facet;
    if (blockIdx.x >= compact_tiles(ncell)) return;
    compact_count_tile(blockIdx.x, C.acc + kAccW * ncell, ncell, C.scan);
}

__global__ __launch_bounds__(kCompactBS) void compact_write_batch_kernel(const BatchDesc *desc,
                                                                          double len)
{
    const unsigned t = blockIdx.y;
    if (t >= desc->ntarget) return;
    const BatchCompact &C = desc->compact[t];
    const unsigned long ncell = (unsigned long)C.facet * C.facet;
    const unsigned nb = compact_tiles(ncell);
    if (blockIdx.x >= nb) return;
    const CompactOut out = C.out;  // in registers: its stores must not reload the descriptor
    compact_write_tile<true>(blockIdx.x, nb, C.acc, C.facet, ncell, len, C.scan, out,
                             C.fx_unscale, C.fs_unscale);
}

void launch_compact_batch(hipStream_t s, const BatchDesc *desc, unsigned ncap, unsigned fmax,
                          double len)
{
    const unsigned nb = compact_tiles((unsigned long)fmax * fmax);
    compact_count_batch_kernel<<<dim3(nb, ncap), kCompactBS, 0, s>>>(desc);
    compact_write_batch_kernel<<<dim3(nb, ncap), kCompactBS, 0, s>>>(desc, len);
}

size_t grid_acc_words(unsigned facet) { return (size_t)kAccWords * facet * facet; }

// ------------------------------------------------------------------ batched extraction
// One persistent pass over the residual for a whole batch (GridBatchLaunch).  A work-group
// takes the next tile of kBatchTileRows sorted rows from the queue; each thread owns 4
// consecutive rows.  Per channel: the thread's visibilities are loaded once, the pending
// updates are applied in order and written back, then every target galaxy grids them with
// the arithmetic of grid_run_kernel (runs of equal cells merged in registers, an LDS table
// of integer sums, flushed to the target's accumulators before the next target).  No
// work-group waits for another, so the launch may hold any number of them; the last one
// to finish leaves the queue counters at zero for the next launch.
template <int PREC>
__global__ __launch_bounds__(256) void grid_batch_kernel(GridBatchLaunch a)
{
    constexpr int BS = 256, RPT = 4, HS = 1024, HBITS = 10;
    static_assert(RPT * BS == kBatchTileRows, "tile rows");
    __shared__ uint32_t hkey[HS];
    __shared__ unsigned long long hre[HS], him[HS], hs2[HS];
    __shared__ uint32_t hcnt[HS];
    __shared__ uint32_t hlist[HS];
    __shared__ uint32_t hn;
    __shared__ unsigned s_tile;
    const int tid = threadIdx.x;
    for (int s = tid; s < HS; s += BS) {
        hkey[s] = kEmpty;
        hre[s] = 0ull;
        him[s] = 0ull;
        hs2[s] = 0ull;
        hcnt[s] = 0;
    }
    if (tid == 0) hn = 0;
    const unsigned ntarget = a.desc->ntarget, nsub = a.desc->nsub;
    while (true) {
        if (tid == 0) s_tile = atomicAdd(&a.queue[0], 1u);
        __syncthreads();
        const unsigned tile = s_tile;
        if (tile >= a.ntiles) break;
        const unsigned long row0 = (unsigned long)tile * kBatchTileRows + (unsigned long)tid * RPT;
        double ru[RPT], rv[RPT], rw[RPT];
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            const unsigned long i = row0 + k;
            const bool in = i < a.nrow;
            ru[k] = in ? a.u[i] : 0.;
            rv[k] = in ? a.v[i] : 0.;
            rw[k] = in ? a.w[i] : 0.;
        }
        for (unsigned c = 0; c < a.nch; c++) {
            const double wn = a.wn[c], inv_lambda = a.inv_lambda[c];
            const double wn2 = wn * wn, spectra = a.spec[c];
            float vs2[RPT];
            double2 vres[RPT];
#pragma unroll
            for (int k = 0; k < RPT; k++) {
                const unsigned long i = row0 + k;
                const size_t idx = (size_t)c * a.nrow + i;
                vs2[k] = i < a.nrow ? a.s2f[idx] : -1.f;
                vres[k] = i < a.nrow ? load_res(a.res, PREC, idx) : make_double2(0., 0.);
            }
            if (nsub) {
                for (unsigned b = 0; b < nsub; b++) {
                    const GalaxyGeom fit = a.desc->subs[b].fit, rnd = a.desc->subs[b].rnd;
#pragma unroll
                    for (int k = 0; k < RPT; k++) {
                        const double p = ru[k] * fit.l0 + rv[k] * fit.m0 + rw[k] * fit.n0;
                        vres[k] = subtract_vis(fit, rnd, p, ru[k], rv[k], wn2, spectra,
                                               inv_lambda, vres[k]);
                        // each update a pass of its own: a complex64 residual is stored
                        // between them
                        if (PREC != 0)
                            vres[k] = make_double2((double)(float)vres[k].x,
                                                   (double)(float)vres[k].y);
                    }
                }
#pragma unroll
                for (int k = 0; k < RPT; k++) {
                    const unsigned long i = row0 + k;
                    if (i >= a.nrow) continue;
                    store_res(a.res, PREC, (size_t)c * a.nrow + i, vres[k]);
                }
            }
            for (unsigned t = 0; t < ntarget; t++) {
                const BatchTarget T = a.desc->targets[t];
                uint32_t rkey = kEmpty, rn = 0;
                long long rre = 0, rim = 0, rs2 = 0;  // integer run sums, as grid_run_kernel
                auto emit = [&](uint32_t key, long long xr, long long xi, long long xs,
                                uint32_t n) {
                    uint32_t h = (key * 2654435761u) >> (32 - HBITS);
                    while (true) {
                        const uint32_t prev = atomicCAS(&hkey[h], kEmpty, key);
                        if (prev == kEmpty) hlist[atomicAdd(&hn, 1u)] = h;
                        if (prev == kEmpty || prev == key) break;
                        h = (h + 1) & (HS - 1);
                    }
                    atomicAdd(&hre[h], (unsigned long long)xr);
                    atomicAdd(&him[h], (unsigned long long)xi);
                    atomicAdd(&hs2[h], (unsigned long long)xs);
                    atomicAdd(&hcnt[h], n);
                };
#pragma unroll
                for (int k = 0; k < RPT; k++) {
                    const unsigned long i = row0 + k;
                    if (i >= a.nrow) continue;
                    const float s2 = vs2[k];
                    if (signbit(s2)) continue;  // flagged
                    const double u = ru[k], v = rv[k];
                    uint32_t key;
                    if (!cell_index_fast(u, v, inv_lambda, a.len, T.inc, T.inv_inc, T.facet, &key))
                        continue;
                    // visGal = round model + residual, shifted by -k(ul + vm + wn)
                    // (source_extraction.c:51-65)
                    const double p = u * T.g.l0 + v * T.g.m0 + rw[k] * T.g.n0;
                    const double shape = model_shape_rsq(T.g, u, v, wn2, spectra);
                    double sn, cs;
                    sincos_rev64(p * inv_lambda, sn, cs);
                    const double gre = shape * cs + vres[k].x;
                    const double gim = shape * sn + vres[k].y;
                    const double xr = gre * cs - gim * (-sn);
                    const double xi = gre * (-sn) + gim * cs;
                    const long long ir = fx_round(xr, T.fx_scale);
                    const long long ii = fx_round(xi, T.fx_scale);
                    const long long is = fx_round((double)s2, a.fs_scale);
                    if (key == rkey) {
                        rre += ir;
                        rim += ii;
                        rs2 += is;
                        rn++;
                    } else {
                        if (rn) emit(rkey, rre, rim, rs2, rn);
                        rkey = key;
                        rre = ir;
                        rim = ii;
                        rs2 = is;
                        rn = 1;
                    }
                }
                if (rn) emit(rkey, rre, rim, rs2, rn);
                __syncthreads();
                const unsigned long ncell = (unsigned long)T.facet * T.facet;
                unsigned long long *acc = (unsigned long long *)T.acc;
                double *acc_w = T.acc + kAccW * ncell;
                const uint32_t nocc = hn;
                for (uint32_t j = tid; j < nocc; j += BS) {
                    const uint32_t s = hlist[j];
                    const uint32_t key = hkey[s];
                    fx_flush(acc + kAccReHi * ncell + key, acc + kAccReLo * ncell + key,
                             (long long)hre[s]);
                    fx_flush(acc + kAccImHi * ncell + key, acc + kAccImLo * ncell + key,
                             (long long)him[s]);
                    fx_flush(acc + kAccS2Hi * ncell + key, acc + kAccS2Lo * ncell + key,
                             (long long)hs2[s]);
                    unsafeAtomicAdd(&acc_w[key], (double)hcnt[s]);
                    hkey[s] = kEmpty;
                    hre[s] = 0ull;
                    him[s] = 0ull;
                    hs2[s] = 0ull;
                    hcnt[s] = 0;
                }
                __syncthreads();
                if (tid == 0) hn = 0;
                __syncthreads();
            }
        }
        __syncthreads();  // every thread has read s_tile before thread 0 takes the next tile
    }
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(&a.queue[1], 1u) == gridDim.x - 1) {
            atomicExch(&a.queue[0], 0u);
            atomicExch(&a.queue[1], 0u);
        }
    }
}

void launch_grid_batch(hipStream_t s, const GridBatchLaunch &a, unsigned groups)
{
    groups = std::max(1u, std::min(groups, a.ntiles));
    if (a.prec == 0)
        grid_batch_kernel<0><<<groups, 256, 0, s>>>(a);
    else
        grid_batch_kernel<1><<<groups, 256, 0, s>>>(a);
}

template <int PREC>
__global__ __launch_bounds__(256) void subtract_batch_kernel(
    unsigned nch, unsigned long nrow, const double *__restrict__ u, const double *__restrict__ v,
    const double *__restrict__ w, const double *__restrict__ wn,
    const double *__restrict__ inv_lambda, const double *__restrict__ spec, const BatchSub *subs,
    unsigned nsub, void *res)
{
    const unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nrow) return;
    const double ui = u[i], vi = v[i], wi = w[i];
    for (unsigned c = 0; c < nch; c++) {
        const double k = wn[c], k2 = k * k, spectra = spec[c];
        const size_t idx = (size_t)c * nrow + i;
        double2 r = load_res(res, PREC, idx);
        for (unsigned b = 0; b < nsub; b++) {
            const GalaxyGeom fit = subs[b].fit, rnd = subs[b].rnd;
            const double p = ui * fit.l0 + vi * fit.m0 + wi * fit.n0;
            r = subtract_vis(fit, rnd, p, ui, vi, k2, spectra, inv_lambda[c], r);
            if (PREC != 0 && b + 1 < nsub)  // each update a pass of its own: stored as complex64
                r = make_double2((double)(float)r.x, (double)(float)r.y);
        }
        store_res(res, PREC, idx, r);
    }
}

void launch_subtract_batch(hipStream_t s, int prec, unsigned nch, unsigned long nrow,
                           const double *u, const double *v, const double *w, const double *wn,
                           const double *inv_lambda, const double *spec, const BatchSub *subs,
                           unsigned nsub, void *res)
{
    if (nsub == 0) return;
    dim3 grid((unsigned)((nrow + 255) / 256));
    if (prec == 0)
        subtract_batch_kernel<0><<<grid, 256, 0, s>>>(nch, nrow, u, v, w, wn, inv_lambda, spec,
                                                      subs, nsub, res);
    else
        subtract_batch_kernel<1><<<grid, 256, 0, s>>>(nch, nrow, u, v, w, wn, inv_lambda, spec,
                                                      subs, nsub, res);
}

// Rows of a gridding work-group (256 threads x rows per thread) for the current variant.
// log2 of the visibilities one LDS slot can receive between flushes: the rows of a
// work-group, times the channels for the variants that keep cells across channels.
// The most terms any gridding path puts in one table slot between flushes, as a power of
// two: 2048 rows (runs of 8), or 1024 rows times every channel (runs of 4 kept across
// channels).  Every path (each variant, the batched kernel) takes its scale from this one
// bound, so their integer sums, and the facets, are the same bit for bit.
static int grid_rows_log2(unsigned nch)
{
    int ch = 0;
    while ((1u << ch) < nch) ch++;
    return std::max(11, 10 + ch);
}

AccScale fx_scales(double vis_bound, double s2_bound, int rows_log2, unsigned nch)
{
    // 2^S with bound * 2^S * (terms a slot takes between flushes) <= 2^62
    if (rows_log2 < 0) rows_log2 = grid_rows_log2(nch);
    auto scale = [&](double b) {
        if (!(b > 0.) || !std::isfinite(b)) b = 1.;
        const int S = std::max(-1000, std::min(1000, 62 - rows_log2 - (ilogb(b) + 1)));
        return ldexp(1.0, S);
    };
    AccScale a;
    a.fx_scale = scale(vis_bound);
    a.fs_scale = scale(s2_bound);
    return a;
}

// Bound max |re| + |im| over the residual (as the bit pattern of a non-negative double, so
// that integer atomicMax orders it).
template <int PREC>
__global__ __launch_bounds__(256) void abs_bound_kernel(const void *res, unsigned long n,
                                                        unsigned long long *out)
{
    double m = 0.;
    const unsigned long step = (unsigned long)gridDim.x * 256ul;
    unsigned long i = blockIdx.x * 256ul + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {
        double2 x[4];
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = load_res(res, PREC, i + k * step);
#pragma unroll
        for (int k = 0; k < 4; k++) m = fmax(m, fabs(x[k].x) + fabs(x[k].y));
    }
    for (; i < n; i += step) {
        const double2 x = load_res(res, PREC, i);
        m = fmax(m, fabs(x.x) + fabs(x.y));
    }
    // one atomic per work-group: on one address they take 12 ns each, and 16,384 of them (one
    // per wave of 4,096 work-groups) took 190 us whatever the residual's size
    __shared__ double part[4];
    for (int off = 32; off >= 1; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmax(fmax(part[0], part[1]), fmax(part[2], part[3]));
        atomicMax(out, (unsigned long long)__double_as_longlong(m));
    }
}

void launch_abs_bound(hipStream_t s, int prec, unsigned long nvis, const void *res,
                      unsigned long long *out)
{
    const unsigned grid = (unsigned)std::min<unsigned long>(2048ul, (nvis + 255) / 256);
    if (prec == 0)
        abs_bound_kernel<0><<<grid, 256, 0, s>>>(res, nvis, out);
    else
        abs_bound_kernel<1><<<grid, 256, 0, s>>>(res, nvis, out);
}

void launch_compact(hipStream_t s, double *acc, unsigned facet, double len, const CompactOut &out,
                    unsigned *scratch, const AccScale *fx)
{
    const unsigned long ncell = (unsigned long)facet * facet;
    const unsigned nb = compact_tiles(ncell);
    // ctr needs a thread per grid index: nb * kCompactBS = ceil(facet^2 / 1024) * 256 >= facet
    // for every facet size
    compact_count_kernel<<<nb, kCompactBS, 0, s>>>(acc + (fx ? kAccW : 3) * ncell, ncell, scratch);
    if (fx)
        compact_write_kernel<true><<<nb, kCompactBS, 0, s>>>(
            acc, facet, ncell, len, scratch, out, 1.0 / fx->fx_scale, 1.0 / fx->fs_scale);
    else
        compact_write_kernel<false><<<nb, kCompactBS, 0, s>>>(acc, facet, ncell, len, scratch, out,
                                                              1.0, 1.0);
}

// ------------------------------------------------------------------ likelihood (K3)
// One work-group per (item, scalelength): the exponential-disk model at zero
// (galaxy_visibilities.c:59-91), the cross-correlation sums and the Newton search of its
// peak (likelihood.c:195-358), and the position marginalisation (likelihood.c:157-187,
// 376-421).  The model normalisation 1/sqrt(sum M^2/sigma^2) is applied at the end: the
// Newton increments are ratios of sums of equal degree in M, so ho = h'/sqrt(S2) and
// det = det'/S2 with h', det' computed from the unnormalised model.
template <int BS, int N>
__device__ inline void block_allreduce(double (&v)[N], double *lds)
{
#pragma unroll
    for (int j = 0; j < N; j++)
        for (int off = 32; off >= 1; off >>= 1) v[j] += __shfl_xor(v[j], off);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int NW = BS / 64;
    if (lane == 0)
#pragma unroll
        for (int j = 0; j < N; j++) lds[wave * N + j] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < N; j++) {
        double t = 0.;
        for (int q = 0; q < NW; q++) t += lds[q * N + j];
        v[j] = t;
    }
    __syncthreads();
}

// Lane values read into scalar registers (l uniform over the wave).
__device__ inline double read_lane(double v, int l)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// Swaps of half rows of two registers: swap32 leaves {a's lanes 0-31, b's lanes 0-31} in a
// and {a's 32-63, b's 32-63} in b; swap16 the same for each pair of rows of 16 lanes.
__device__ inline void swap32(double &a, double &b)
{
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false,
                                                    false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false,
                                                    false);
    a = __hiloint2double((int)h[0], (int)l[0]);
    b = __hiloint2double((int)h[1], (int)l[1]);
}
__device__ inline void swap16(double &a, double &b)
{
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false,
                                                    false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false,
                                                    false);
    a = __hiloint2double((int)h[0], (int)l[0]);
    b = __hiloint2double((int)h[1], (int)l[1]);
}
// A lane permutation within rows that every lane takes part in.
template <int CTRL>
__device__ inline double dpp_perm_f64(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int rlo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, true);
    const int rhi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, true);
    return __hiloint2double(rhi, rlo);
}

// Shifts over the whole wave by one lane (0x138 wave_shr:1: from the lane before, 0x130
// wave_shl:1: from the lane after); 0 where there is none.
template <int CTRL>
__device__ inline double dpp_shift_f64(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int rlo = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true);
    const int rhi = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true);
    return __hiloint2double(rhi, rlo);
}

// Each lane's value of the lane whose number differs in bit 2 (the other half of its eight):
// shifts by 4 into the banks of four lanes that have a source in their half.
__device__ inline double dpp_xor4_f64(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    int rlo = __builtin_amdgcn_update_dpp(lo, lo, 0x104, 0xf, 0x5, false);  // row_shl:4
    int rhi = __builtin_amdgcn_update_dpp(hi, hi, 0x104, 0xf, 0x5, false);
    rlo = __builtin_amdgcn_update_dpp(rlo, lo, 0x114, 0xf, 0xa, false);  // row_shr:4
    rhi = __builtin_amdgcn_update_dpp(rhi, hi, 0x114, 0xf, 0xa, false);
    return __hiloint2double(rhi, rlo);
}

// The sum of v over the eight lanes with the same lane % 8, in each of them.
__device__ inline double wave_sum_by8(double v)
{
    v += dpp_perm_f64<0x128>(v);  // row_ror:8
    double w = v;
    swap16(v, w);
    v += w;
    w = v;
    swap32(v, w);
    return v + w;
}

// The wave's sum in every lane, by data-parallel-primitive moves (lane shifts in the VALU, no
// LDS round trips): the lanes are paired by bit 0 of their number, then bit 1, and so on, a
// fixed order, and both lanes of a pair get the same bits.  Read into scalar registers, so
// that the wave takes the same branches after it.
__device__ inline double wave_sum(double v)
{
    v += dpp_perm_f64<0xb1>(v);  // quad_perm [1, 0, 3, 2]
    v += dpp_perm_f64<0x4e>(v);  // quad_perm [2, 3, 0, 1]
    v += dpp_xor4_f64(v);
    return read_lane(wave_sum_by8(v), 0);
}

// The wave's sums of eight values at once: the total of v[lane % 8] in every lane.  The lanes
// are paired as in wave_sum (the same bits), but each of the first three steps also halves the
// number of values that a lane holds: 10 additions with their moves instead of 48.  The seven
// sums of a work-group one after the other took 900 cycles of a Newton pass of 5,700, and those
// of the task's chunks as much again; with this the loop over 24 galaxies of a 64-dish array
// went from 26.3 to 24.7 ms, batches of 16 (48 galaxies) from 15.1 to 10.5 ms, 63 points on 496
// cells from 70.8 to 57.1 us, and 4 points on 72,000 cells from 100.5 to 97.0 us.
__device__ inline double wave_sum8(const double (&v)[8])
{
    const int lane = threadIdx.x & 63;
    double w[4], x[2];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const double keep = lane & 1 ? v[2 * k + 1] : v[2 * k];
        w[k] = keep + dpp_perm_f64<0xb1>(lane & 1 ? v[2 * k] : v[2 * k + 1]);  // quad_perm 1032
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const double keep = lane & 2 ? w[2 * k + 1] : w[2 * k];
        x[k] = keep + dpp_perm_f64<0x4e>(lane & 2 ? w[2 * k] : w[2 * k + 1]);  // quad_perm 2301
    }
    const double keep = lane & 4 ? x[1] : x[0];
    return wave_sum_by8(keep + dpp_xor4_f64(lane & 4 ? x[0] : x[1]));
}

// The wave's maximum in every lane, paired as in wave_sum.  fmax is exact (and skips NaN), so
// the result does not depend on the order.
__device__ inline double wave_max(double v)
{
    v = fmax(v, dpp_perm_f64<0xb1>(v));
    v = fmax(v, dpp_perm_f64<0x4e>(v));
    v = fmax(v, dpp_xor4_f64(v));
    v = fmax(v, dpp_perm_f64<0x128>(v));
    double w = v;
    swap16(v, w);
    v = fmax(v, w);
    w = v;
    swap32(v, w);
    return read_lane(fmax(v, w), 0);
}

// expint_ei (rl2_math.h) of two arguments by one wave, the same bits: the divisions of up to 64
// terms are made by the lanes at once, and only the products and the sums that the series
// carry from term to term run one after the other, on two lanes (one argument each) through
// LDS.  One lane's series took two divisions a term, a hundred terms at the longest: with the
// series on one lane the loop over 24 galaxies of a 64-dish array took 45.0 ms, with this
// 38.5 (prefix products over the lanes took no longer, but round differently, and where few
// points are sampled a last bit decides whether a variance is a number).
// x0, x1 > 0 and the same in every lane; one wave of a work-group at a time (buf).
__device__ __attribute__((always_inline)) inline void expint_ei_wave(double x0, double x1, double *y0, double *y1)
{
    const double euler = 0.57721566490153286060651209008240243;
    constexpr int U = 8;
    __shared__ double buf[2][64 + U];
    const int lane = threadIdx.x & 63;
    const bool as0 = !(x0 <= 40.), as1 = !(x1 <= 40.);  // asymptotic series
    const double *mine = buf[lane & 1];
    double *put = buf[lane & 1];
    // the recurrences over buf[0] and buf[1] in place, by lanes 0 and 1: c = op(c, buf[i])
    auto chain = [&](int steps, double c, auto op) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < 2) {
            // two sets of U values, each read while the other is used (past the last: the
            // buffer's tail); no copies between them, which would wait for the reads
            double v[U], w[U];
            auto use = [&](const double (&x)[U], int i) {
#pragma unroll
                for (int j = 0; j < U; j++) {
                    c = op(c, x[j]);
                    put[i + j] = c;
                }
            };
            auto read = [&](double (&x)[U], int i) {
#pragma unroll
                for (int j = 0; j < U; j++) x[j] = mine[i + j];
            };
            read(v, 0);
            for (int i = 0; i < steps; i += 2 * U) {
                read(w, i + U);
                use(v, i);
                read(v, i + 2 * U);
                use(w, i + U);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        return c;
    };
    double term = 1., sum = (lane & 1 ? as1 : as0) ? 1. : 0.;  // lanes 0 and 1: carried
    double s0 = 0., s1 = 0.;
    bool done0 = false, done1 = false;
    for (int base = 0; base < 1024 && !(done0 && done1); base += 64) {
        const int steps =
            min(64, ((int)(2.2 * fmin(fmax(x0, x1), 40.)) + 24 + 2 * U - 1) / (2 * U) * (2 * U));
        const double k = (double)(base + lane + 1);
        buf[0][lane] = as0 ? k / x0 : x0 / k;
        buf[1][lane] = as1 ? k / x1 : x1 / k;
        const double t_in = term;
        term = chain(steps, term, [](double c, double v) { return c * v; });
        const double p0 = buf[0][lane], p1 = buf[1][lane];
        const double q0 = lane ? buf[0][lane - 1] : read_lane(t_in, 0);
        const double q1 = lane ? buf[1][lane - 1] : read_lane(t_in, 1);
        const double t0 = as0 ? p0 : p0 / k, t1 = as1 ? p1 : p1 / k;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        buf[0][lane] = t0;
        buf[1][lane] = t1;
        const double s_in = sum;
        sum = chain(steps, sum, [](double c, double v) { return c + v; });
        // the first term at which the series ends: with it (below eps / 4 of the sum), or
        // before it (an asymptotic term no smaller than the one before)
        auto end = [&](const double *S, double t, double q, bool as, double in, double *s) {
            const double sl = S[lane];
            const bool before = as && t >= q;
            const uint64_t m =
                __ballot(lane < steps && (before || t < 2.220446049250313e-16 * 0.25 * sl));
            const int f = m ? __ffsll((unsigned long long)m) - 1 : steps - 1;
            const bool b = m && ((__ballot(before) >> f) & 1);
            *s = b ? (f ? read_lane(sl, f - 1) : in) : read_lane(sl, f);
            return m != 0;
        };
        double s;
        const bool e0 = end(buf[0], t0, q0, as0, read_lane(s_in, 0), &s);
        if (!done0) s0 = s;
        done0 = done0 || e0;
        const bool e1 = end(buf[1], t1, q1, as1, read_lane(s_in, 1), &s);
        if (!done1) s1 = s;
        done1 = done1 || e1;
        if (steps < 64 && !(done0 && done1)) base -= 64 - steps;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    *y0 = as0 ? exp(x0) / x0 * s0 : euler + log(x0) + s0;
    *y1 = as1 ? exp(x1) / x1 * s1 : euler + log(x1) + s1;
}

// marg_position (rl2_math.h) by a wave, for an argument that is the same in all its lanes,
// with the same bits.  The two exponential integrals of a task that ends with B <= 100 were its
// longest serial chain, by one lane, on the critical path of the Newton pass.
__device__ __attribute__((always_inline)) inline double marg_position_wave(double x)
{
    const double Delta = 0.5 * 5.991;
    if (x <= Delta) return kBad;
    if (x > 100.) return x - log(Delta) - exp(-Delta);
    if ((x - Delta) < 0.0001) x = Delta + 0.0001;
    double yc, ys;
    expint_ei_wave(x, x - Delta, &yc, &ys);
    return log((yc - ys) / log(x / (x - Delta)));
}

// likelihood.c:174-183: L_r = log of the position-marginalised likelihood minus
// 1/2 log det of the cross-correlation Hessian; -1e10 when the peak search failed.  Called
// by a whole wave with the same arguments in every lane; lane 0 writes.
__device__ __attribute__((always_inline)) inline void finish_lr(const LikLaunch &a, int item, int r, double ho,
                                 double det_sigma, int iter)
{
    double L;
    if (det_sigma <= 0)
        L = kBad;
    else {
        const double B = (ho * ho) * 0.5;
        L = marg_position_wave(B);
        if (isnan(L))
            L = kBad;
        else
            L -= 0.5 * log(det_sigma);
    }
    if ((threadIdx.x & 63) != 0) return;
    // at agent scope: the small-facet kernel's last work-group of an item reads it
    __hip_atomic_store(a.Lr + (size_t)item * kMaxR + r, L, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    a.nit[(size_t)item * kMaxR + r] = iter;
    if (a.Lr_host) {  // pinned memory, where the host polls for them or reads them at the end
        a.Lr_host[(size_t)item * kMaxR + r] = L;
        a.nit_host[(size_t)item * kMaxR + r] = iter;
    }
    if (a.ho) a.ho[(size_t)item * kMaxR + r] = ho;
    if (a.det) a.det[(size_t)item * kMaxR + r] = det_sigma;
}

template <int BS, int PPT>
__global__ __launch_bounds__(BS) void likelihood_kernel(LikLaunch a)
{
    __shared__ double red[(BS / 64) * 8];
    const int nr = a.rg.numr - 1;
    const int item = blockIdx.x / nr;
    const int r = blockIdx.x % nr + 1;
    const LikItem it = a.items[item];
    if (it.prec != 0) return;  // evaluated by the mixed-precision kernel
    const FacetDev &F = a.facets[it.slot];
    const unsigned n = F.n;
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(a.rg.ro[r]);
    const double sf = (scale * scale) / (detA * detA);
    const double cc2 = 4 * kPi * kPi;
    const double sw = sf * cc2;
    const double a1 = 1. + e1, a2 = 1. - e1;
    const double *__restrict__ gu = F.uu;
    const double *__restrict__ gv = F.vv;
    const double *__restrict__ dre = F.dre;
    const double *__restrict__ dim = F.dim;
    const double *__restrict__ gs2 = F.s2;
    const double *__restrict__ gmod = F.mod;
    const int tid = threadIdx.x;

    // Point terms of the first PPT*BS cells stay in registers (static indices so the
    // cache is not demoted to scratch memory); cells beyond are recomputed per pass.
    double hrc[PPT > 0 ? PPT : 1], hic[PPT > 0 ? PPT : 1];
    double s[7] = {0., 0., 0., 0., 0., 0., 0.};  // S2, value, dx, dy, dxx, dyy, dxy
    // (1 + s w |k|^2)^(-3/2) as rsqrt(den)^3: one reciprocal square root instead of a
    // square root and a division (a few ulp from the reference's 1/(den*sqrt(den))).
    auto model_at = [&](unsigned i, double uu, double vv) -> double {
        if (gmod) return gmod[i];
        const double k1 = a1 * uu + e2 * vv;
        const double k2 = e2 * uu + a2 * vv;
        const double rr = rsqrt(1. + sw * (k1 * k1 + k2 * k2));
        return rr * rr * rr;
    };
    auto pass0 = [&](unsigned i, double &hr, double &hi) {
        const double uu = gu[i], vv = gv[i];
        const double M = model_at(i, uu, vv);
        s[0] += M * M / gs2[i];
        hr = dre[i] * M;
        hi = -dim[i] * M;
        const double U = kTwoPi * uu, V = kTwoPi * vv;
        s[1] += hr;
        s[2] -= hi * U;
        s[3] -= hi * V;
        s[4] -= hr * U * U;
        s[5] -= hr * V * V;
        s[6] -= hr * U * V;
    };
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const unsigned i = tid + k * BS;
        hrc[k] = 0.;
        hic[k] = 0.;
        if (i < n) pass0(i, hrc[k], hic[k]);
    }
    for (unsigned i = tid + PPT * BS; i < n; i += BS) {
        double hr, hi;
        pass0(i, hr, hi);
    }
    block_allreduce<BS, 7>(s, red);
    const double S2 = gmod ? 1.0 : s[0];
    double value = s[1], dx = s[2], dy = s[3], dxx = s[4], dyy = s[5], dxy = s[6];
    double det = dxx * dyy - dxy * dxy;
    double xo = 0., yo = 0., norm = 1.;
    int iter = 0;
    while (det > 0 && norm > 1.e-7 && iter < 50) {
        iter++;
        const double incx = (dx * dyy - dy * dxy) / det;
        const double incy = (dy * dxx - dx * dxy) / det;
        xo -= incx;
        yo -= incy;
        double t[6] = {0., 0., 0., 0., 0., 0.};
        auto newton_term = [&](unsigned i, double hr, double hi) {
            const double U = kTwoPi * gu[i], V = kTwoPi * gv[i];
            const double ph = xo * U + yo * V;
            double sn, cs;
            sincos(ph, &sn, &cs);
            const double re = hr * cs - hi * sn;
            const double im = hr * sn + hi * cs;
            t[0] += re;
            t[1] -= im * U;
            t[2] -= im * V;
            t[3] -= re * U * U;
            t[4] -= re * V * V;
            t[5] -= re * U * V;
        };
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            const unsigned i = tid + k * BS;
            if (i < n) newton_term(i, hrc[k], hic[k]);
        }
        for (unsigned i = tid + PPT * BS; i < n; i += BS) {
            const double M = model_at(i, gu[i], gv[i]);
            newton_term(i, dre[i] * M, -dim[i] * M);
        }
        block_allreduce<BS, 6>(t, red);
        value = t[0];
        dx = t[1];
        dy = t[2];
        dxx = t[3];
        dyy = t[4];
        dxy = t[5];
        det = dxx * dyy - dxy * dxy;
        norm = sqrt(incx * incx + incy * incy);
    }
    if (tid < 64)
        finish_lr(a, item, r, gmod ? value : value / sqrt(S2), gmod ? det : det / S2, iter);
}

// ------------------------------------------------------------------ likelihood, mixed
// FP32 model and cross-correlation terms from the packed facet {u, v, D_re, D_im}; the
// Newton phase x.u + y.v is formed and reduced in FP64 (revolutions), sin/cos evaluated
// in FP32 on the reduced octant; per-thread partial sums are flushed to FP64 every
// kFlush cells; the Newton update, position and scalelength marginalisation run in FP64.
constexpr int kFlush = 8;

// sin(2 pi t), cos(2 pi t): t reduced to [-1/2, 1/2] in FP64, then to an octant
// |y| <= 1/8 in FP32; Taylor series of sin / cos of 2 pi y to degree 9 / 10
// (truncation < 3e-9 on the octant).
__device__ inline void sincos_rev(double t, float &sn, float &cs)
{
    const float x = (float)(t - rint(t));
    const float q = rintf(4.f * x);
    const float y = x - 0.25f * q;
    const float th = 6.28318530717958648f * y;
    const float z = th * th;
    const float ps = fmaf(fmaf(fmaf(1.f / 362880, z, -1.f / 5040), z, 1.f / 120), z, -1.f / 6);
    const float s = fmaf(th * z, ps, th);
    const float pc = fmaf(fmaf(fmaf(fmaf(-1.f / 3628800, z, 1.f / 40320), z, -1.f / 720), z,
                               1.f / 24), z, -0.5f);
    const float c = fmaf(pc, z, 1.f);
    const int k = ((int)q) & 3;
    sn = (k == 0) ? s : (k == 1) ? c : (k == 2) ? -s : -c;
    cs = (k == 0) ? c : (k == 1) ? -s : (k == 2) ? -c : s;
}

template <int BS, int PPT>
__global__ __launch_bounds__(BS) void likelihood32_kernel(LikLaunch a)
{
    __shared__ double red[(BS / 64) * 8];
    const int nr = a.rg.numr - 1;
    const int item = blockIdx.x / nr;
    const int r = blockIdx.x % nr + 1;
    const LikItem it = a.items[item];
    if (it.prec != 1) return;
    const FacetDev &F = a.facets[it.slot];
    const unsigned n = F.n;
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(a.rg.ro[r]);
    const double sf = (scale * scale) / (detA * detA);
    const float sw = (float)(sf * (4 * kPi * kPi));
    const float a1 = (float)(1. + e1), a2 = (float)(1. - e1), fe2 = (float)e2;
    const float tp = 6.28318530717958648f;
    const float4 *__restrict__ pk = F.pk;
    const float *__restrict__ is2 = F.invs2;
    const int tid = threadIdx.x;

    float hrc[PPT > 0 ? PPT : 1], hic[PPT > 0 ? PPT : 1];
    double s[7] = {0., 0., 0., 0., 0., 0., 0.};
    float f[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int cnt = 0;
    auto model = [&](const float4 p) -> float {
        const float k1 = a1 * p.x + fe2 * p.y;
        const float k2 = fe2 * p.x + a2 * p.y;
        const float rr = rsqrtf(1.f + sw * (k1 * k1 + k2 * k2));
        return rr * rr * rr;
    };
    auto flush7 = [&]() {
#pragma unroll
        for (int j = 0; j < 7; j++) {
            s[j] += (double)f[j];
            f[j] = 0.f;
        }
    };
    auto pass0 = [&](unsigned i, float &hr, float &hi) {
        const float4 p = pk[i];
        const float M = model(p);
        hr = p.z * M;
        hi = -p.w * M;
        const float U = tp * p.x, V = tp * p.y;
        f[0] += M * M * is2[i];
        f[1] += hr;
        f[2] -= hi * U;
        f[3] -= hi * V;
        f[4] -= hr * U * U;
        f[5] -= hr * V * V;
        f[6] -= hr * U * V;
        if (++cnt == kFlush) {
            flush7();
            cnt = 0;
        }
    };
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const unsigned i = tid + k * BS;
        hrc[k] = 0.f;
        hic[k] = 0.f;
        if (i < n) pass0(i, hrc[k], hic[k]);
    }
    for (unsigned i = tid + PPT * BS; i < n; i += BS) {
        float hr, hi;
        pass0(i, hr, hi);
    }
    flush7();
    block_allreduce<BS, 7>(s, red);
    const double S2 = s[0];
    double value = s[1], dx = s[2], dy = s[3], dxx = s[4], dyy = s[5], dxy = s[6];
    double det = dxx * dyy - dxy * dxy;
    double xo = 0., yo = 0., norm = 1.;
    int iter = 0;
    while (det > 0 && norm > 1.e-7 && iter < 50) {
        iter++;
        const double incx = (dx * dyy - dy * dxy) / det;
        const double incy = (dy * dxx - dx * dxy) / det;
        xo -= incx;
        yo -= incy;
        double t[6] = {0., 0., 0., 0., 0., 0.};
        float g[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        cnt = 0;
        auto newton_term = [&](const float4 p, float hr, float hi) {
            float sn, cs;
            sincos_rev(xo * (double)p.x + yo * (double)p.y, sn, cs);
            const float U = tp * p.x, V = tp * p.y;
            const float re = hr * cs - hi * sn;
            const float im = hr * sn + hi * cs;
            g[0] += re;
            g[1] -= im * U;
            g[2] -= im * V;
            g[3] -= re * U * U;
            g[4] -= re * V * V;
            g[5] -= re * U * V;
            if (++cnt == kFlush) {
#pragma unroll
                for (int j = 0; j < 6; j++) {
                    t[j] += (double)g[j];
                    g[j] = 0.f;
                }
                cnt = 0;
            }
        };
#pragma unroll
        for (int k = 0; k < PPT; k++) {
            const unsigned i = tid + k * BS;
            if (i < n) newton_term(pk[i], hrc[k], hic[k]);
        }
        for (unsigned i = tid + PPT * BS; i < n; i += BS) {
            const float4 p = pk[i];
            const float M = model(p);
            newton_term(p, p.z * M, -p.w * M);
        }
#pragma unroll
        for (int j = 0; j < 6; j++) t[j] += (double)g[j];
        block_allreduce<BS, 6>(t, red);
        value = t[0];
        dx = t[1];
        dy = t[2];
        dxx = t[3];
        dyy = t[4];
        dxy = t[5];
        det = dxx * dyy - dxy * dxy;
        norm = sqrt(incx * incx + incy * incy);
    }
    if (tid < 64) finish_lr(a, item, r, value / sqrt(S2), det / S2, iter);
}

void launch_likelihood(hipStream_t s, const LikLaunch &a)
{
    if (a.nitems <= 0) return;
    dim3 grid((unsigned)(a.nitems * (a.rg.numr - 1)));
    bool any64 = false, any32 = false;
    for (int i = 0; i < a.nitems; i++) {  // host copy of the request precisions
        if (a.host_prec && a.host_prec[i]) any32 = true; else any64 = true;
    }
    if (any64) {
        switch (a.block) {
        // PPT: register-cached cells per thread; larger caches spill FP64 sincos state.
        case 64: likelihood_kernel<64, 4><<<grid, 64, 0, s>>>(a); break;
        case 128: likelihood_kernel<128, 4><<<grid, 128, 0, s>>>(a); break;
        case 512: likelihood_kernel<512, 0><<<grid, 512, 0, s>>>(a); break;
        case 1024: likelihood_kernel<1024, 0><<<grid, 1024, 0, s>>>(a); break;
        default: likelihood_kernel<256, 4><<<grid, 256, 0, s>>>(a); break;
        }
    }
    if (any32) {
        switch (a.block) {
        case 128: likelihood32_kernel<128, 8><<<grid, 128, 0, s>>>(a); break;
        case 512: likelihood32_kernel<512, 4><<<grid, 512, 0, s>>>(a); break;
        case 1024: likelihood32_kernel<1024, 2><<<grid, 1024, 0, s>>>(a); break;
        default: likelihood32_kernel<256, 8><<<grid, 256, 0, s>>>(a); break;
        }
    }
}

// The FP32 and packed copies of a facet given by a caller (compaction writes an extracted one's).
__global__ void pack_facet_kernel(unsigned n, const double *uu, const double *vv,
                                  const double *dre, const double *dim, const double *s2,
                                  float4 *pk, float *invs2, double *invs2_64, double2 *dc)
{
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        pk[i] = make_float4((float)uu[i], (float)vv[i], (float)dre[i], (float)dim[i]);
        const double w = 1.0 / s2[i];
        invs2[i] = (float)w;
        invs2_64[i] = w;
        pack_cell_records(i, dre[i], dim[i], nullptr, 0u, 0u, dc, nullptr);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {  // the zero pad cell
        invs2_64[n] = 0.;
        pack_cell_records(n, 0., 0., nullptr, 0u, 0u, dc, nullptr);
    }
}

void launch_pack_facet(hipStream_t s, unsigned n, const double *uu, const double *vv,
                       const double *dre, const double *dim, const double *s2, float4 *pk,
                       float *invs2, double *invs2_64, double2 *dc)
{
    const unsigned blocks = std::min(2048u, (n + 255) / 256 + 1);
    pack_facet_kernel<<<blocks, 256, 0, s>>>(n, uu, vv, dre, dim, s2, pk, invs2, invs2_64, dc);
}

// ------------------------------------------------------------------ r-marginalisation (K4)
// One thread per item: set_posterior_values (marginalise_r.c:29-64), then the spline +
// QAG-GK41 integral of marginalise_posterior_r (marginalise_r.c:81-223).
struct QagWs {
    double *alist, *blist, *rlist, *elist;
    int *order, *level;
};

// QUADPACK's error rescaling (GSL 2.5 err.c).  (200 err / asc)^1.5 is formed as x sqrt(x):
// within 1.5 ulp of the correctly rounded power (sqrt is correctly rounded), an order of
// magnitude fewer instructions than pow on the r-marginalisation's serial chain, and the
// value only feeds comparisons with tolerances.
__device__ inline double rescale_error(double err, double result_abs, double result_asc)
{
    err = fabs(err);
    if (result_asc != 0 && err != 0) {
        const double x = 200 * err / result_asc;
        double scale = x * sqrt(x);
        err = (scale < 1) ? result_asc * scale : result_asc;
    }
    if (result_abs > kDblMin / (50 * kDblEps)) {
        double min_err = 50 * kDblEps * result_abs;
        if (min_err > err) err = min_err;
    }
    return err;
}

__device__ inline void qk41_spline(const Spline &sp, double a, double b, double *result,
                                   double *abserr, double *resabs, double *resasc)
{
    const int n = 21;
    double fv1[21], fv2[21];
    const double center = 0.5 * (a + b);
    const double half_length = 0.5 * (b - a);
    const double abs_half_length = fabs(half_length);
    const double f_center = spline_exp(sp, center);
    double result_gauss = 0;
    double result_kronrod = f_center * kWgk41[n - 1];
    double result_abs = fabs(result_kronrod);
    for (int j = 0; j < (n - 1) / 2; j++) {
        const int jtw = j * 2 + 1;
        const double abscissa = half_length * kXgk41[jtw];
        const double f1 = spline_exp(sp, center - abscissa);
        const double f2 = spline_exp(sp, center + abscissa);
        const double fsum = f1 + f2;
        fv1[jtw] = f1;
        fv2[jtw] = f2;
        result_gauss += kWg41[j] * fsum;
        result_kronrod += kWgk41[jtw] * fsum;
        result_abs += kWgk41[jtw] * (fabs(f1) + fabs(f2));
    }
    for (int j = 0; j < n / 2; j++) {
        const int jtwm1 = j * 2;
        const double abscissa = half_length * kXgk41[jtwm1];
        const double f1 = spline_exp(sp, center - abscissa);
        const double f2 = spline_exp(sp, center + abscissa);
        fv1[jtwm1] = f1;
        fv2[jtwm1] = f2;
        result_kronrod += kWgk41[jtwm1] * (f1 + f2);
        result_abs += kWgk41[jtwm1] * (fabs(f1) + fabs(f2));
    }
    const double mean = result_kronrod * 0.5;
    double result_asc = kWgk41[n - 1] * fabs(f_center - mean);
    for (int j = 0; j < n - 1; j++)
        result_asc += kWgk41[j] * (fabs(fv1[j] - mean) + fabs(fv2[j] - mean));
    const double err = (result_kronrod - result_gauss) * half_length;
    result_kronrod *= half_length;
    result_abs *= abs_half_length;
    result_asc *= abs_half_length;
    *result = result_kronrod;
    *resabs = result_abs;
    *resasc = result_asc;
    *abserr = rescale_error(err, result_abs, result_asc);
}

// QUADPACK qpsrt: keep the error list descending
__device__ inline void qpsrt(QagWs &w, int size, int limit, int &nrmax, int &imax)
{
    const int last = size - 1;
    int i_nrmax = nrmax;
    int i_maxerr = w.order[i_nrmax];
    if (last < 2) {
        w.order[0] = 0;
        w.order[1] = 1;
        imax = i_maxerr;
        return;
    }
    const double errmax = w.elist[i_maxerr];
    while (i_nrmax > 0 && errmax > w.elist[w.order[i_nrmax - 1]]) {
        w.order[i_nrmax] = w.order[i_nrmax - 1];
        i_nrmax--;
    }
    int top = (last < (limit / 2 + 2)) ? last : limit - last + 1;
    int i = i_nrmax + 1;
    while (i < top && errmax < w.elist[w.order[i]]) {
        w.order[i - 1] = w.order[i];
        i++;
    }
    w.order[i - 1] = i_maxerr;
    const double errmin = w.elist[last];
    int k = top - 1;
    while (k > i - 2 && errmin >= w.elist[w.order[k]]) {
        w.order[k + 1] = w.order[k];
        k--;
    }
    w.order[k + 1] = last;
    imax = w.order[i_nrmax];
    nrmax = i_nrmax;
}

// gsl_integration_qag semantics (GSL 2.5 qag.c) with the 41-point rule; 0 = success.
__device__ int qag41_spline(const Spline &sp, double a, double b, double epsrel, int limit,
                            QagWs &w, double *result)
{
    double result0, abserr0, resabs0, resasc0;
    int roundoff_type1 = 0, roundoff_type2 = 0, error_type = 0;
    w.alist[0] = a;
    w.blist[0] = b;
    w.rlist[0] = 0.0;
    w.elist[0] = 0.0;
    w.order[0] = 0;
    w.level[0] = 0;
    int size = 0, nrmax = 0, imax = 0;
    *result = 0;
    qk41_spline(sp, a, b, &result0, &abserr0, &resabs0, &resasc0);
    size = 1;
    w.rlist[0] = result0;
    w.elist[0] = abserr0;
    double tolerance = fmax(0., epsrel * fabs(result0));
    const double round_off = 50 * kDblEps * resabs0;
    if (abserr0 <= round_off && abserr0 > tolerance) {
        *result = result0;
        return 14;
    } else if ((abserr0 <= tolerance && abserr0 != resasc0) || abserr0 == 0.0) {
        *result = result0;
        return 0;
    } else if (limit == 1) {
        *result = result0;
        return 11;
    }
    double area = result0, errsum = abserr0;
    int iteration = 1;
    do {
        const double a_i = w.alist[imax], b_i = w.blist[imax];
        const double r_i = w.rlist[imax], e_i = w.elist[imax];
        const double a1 = a_i, b1 = 0.5 * (a_i + b_i), a2 = b1, b2 = b_i;
        double area1, area2, error1, error2, resabs1, resabs2, resasc1, resasc2;
        qk41_spline(sp, a1, b1, &area1, &error1, &resabs1, &resasc1);
        qk41_spline(sp, a2, b2, &area2, &error2, &resabs2, &resasc2);
        const double area12 = area1 + area2;
        const double error12 = error1 + error2;
        errsum += (error12 - e_i);
        area += area12 - r_i;
        if (resasc1 != error1 && resasc2 != error2) {
            const double delta = r_i - area12;
            if (fabs(delta) <= 1.0e-5 * fabs(area12) && error12 >= 0.99 * e_i) roundoff_type1++;
            if (iteration >= 10 && error12 > e_i) roundoff_type2++;
        }
        tolerance = fmax(0., epsrel * fabs(area));
        if (errsum > tolerance) {
            if (roundoff_type1 >= 6 || roundoff_type2 >= 20) error_type = 2;
            const double tmp = (1 + 100 * kDblEps) * (fabs(a2) + 1000 * kDblMin);
            if (fabs(a1) <= tmp && fabs(b2) <= tmp) error_type = 3;
        }
        // update(): bisected halves, larger error first in place
        const int i_max = imax, i_new = size;
        const int new_level = w.level[i_max] + 1;
        if (error2 > error1) {
            w.alist[i_max] = a2;
            w.rlist[i_max] = area2;
            w.elist[i_max] = error2;
            w.level[i_max] = new_level;
            w.alist[i_new] = a1;
            w.blist[i_new] = b1;
            w.rlist[i_new] = area1;
            w.elist[i_new] = error1;
            w.level[i_new] = new_level;
        } else {
            w.blist[i_max] = b1;
            w.rlist[i_max] = area1;
            w.elist[i_max] = error1;
            w.level[i_max] = new_level;
            w.alist[i_new] = a2;
            w.blist[i_new] = b2;
            w.rlist[i_new] = area2;
            w.elist[i_new] = error2;
            w.level[i_new] = new_level;
        }
        size++;
        qpsrt(w, size, limit, nrmax, imax);
        iteration++;
    } while (iteration < limit && !error_type && errsum > tolerance);
    double sum = 0;
    for (int k = 0; k < size; k++) sum += w.rlist[k];
    *result = sum;
    if (errsum <= tolerance) return 0;
    if (error_type == 2) return 14;
    if (error_type == 3) return 21;
    if (iteration == limit) return 11;
    return 5;
}

// marginalise_r.c:81-223 on (num, x, y); y is modified (y -= ymax).
__device__ double marginalise_posterior(int num, const double *x, double *y, QagWs &w)
{
    double ymax = -10.0;
    int ymaxpos = 0;
    for (int ii = 0; ii < num; ii++)
        if (y[ii] > ymax) {
            ymax = y[ii];
            ymaxpos = ii;
        }
    double xmin = x[ymaxpos], xmax = x[ymaxpos];
    if (ymaxpos < num - 1) xmax = x[ymaxpos + 1];
    if (ymaxpos > 0) xmin = x[ymaxpos - 1];
    for (int ii = 0; ii < num; ii++) {
        if (x[ii] < xmin) xmin = x[ii];
        if (x[ii] > xmax) xmax = x[ii];
        y[ii] -= ymax;
    }
    if (xmax <= xmin) return NAN;
    Spline sp;
    double sump = 0.;
    if (spline_init(sp, x, y, num, 0)) return NAN;
    int st = qag41_spline(sp, xmin, xmax, 1.e-3, kQagLimit, w, &sump);
    if (st) {
        spline_init(sp, x, y, num, 1);
        st = qag41_spline(sp, xmin, xmax, 1.e-3, kQagLimit, w, &sump);
    }
    if (st) return kBad;
    return log(sump) + ymax;
}

// Wave-cooperative variants: one work-group of two waves per item.  Lane j of a wave
// evaluates the integrand at Gauss-Kronrod node j (0..19 left of the centre, 20..39 right,
// 40 the centre) and contributes its weighted terms to the Kronrod, Gauss, |f| and
// |f - mean| sums, which wave_sum completes; every lane ends with the same sums (lane
// 63's, read into scalar registers), so all lanes follow the same control flow.  The sums
// differ from QUADPACK's sequential order only by rounding.  Each bisection integrates its
// two halves on the two waves at once.

// The spline of the r-marginalisation in LDS with the cubic coefficients b_i and d_i of each
// interval (cspline_eval's), formed once per spline: spline_exp_lds then takes no division
// per evaluation and, as b_i and d_i are the same expressions of the same knot data, gives
// spline_exp's values bit for bit.
struct SplineLds {
    Spline s;
    double b[kMaxR], d[kMaxR];
};

// The interval is found by counting the inner knots at or below x: with strictly increasing
// knots (spline_build_wave checks them) that is the index cspline_eval's bisection finds, and
// the reads are independent of each other rather than a chain of dependent LDS round trips.
__device__ inline double spline_exp_lds(const SplineLds &t, double x)
{
    const Spline &s = t.s;
    const int n = s.n;
    if (x < s.x[0] || x > s.x[n - 1]) return 0.;
    int lo = 0;
#pragma unroll 8
    for (int j = 1; j < n - 1; j++) lo += s.x[j] <= x ? 1 : 0;
    const double x_lo = s.x[lo], x_hi = s.x[lo + 1];
    const double dx = x_hi - x_lo;
    if (!(dx > 0.0)) return 0.;
    const double y_lo = s.y[lo];
    double y;
    if (s.linear) {
        y = y_lo + (x - x_lo) / dx * (s.y[lo + 1] - y_lo);
    } else {
        const double delx = x - x_lo;
        y = y_lo + delx * (t.b[lo] + delx * (s.c[lo] + delx * t.d[lo]));
    }
    return exp(y);
}

// What the r-marginalisation reads of an item besides its L_r; a lane holds scalelength index
// `lane`'s prior and the Gauss-Kronrod node of that number, and row `lane` of the factored
// spline system of the whole grid.
struct Gk41Node {
    double x, wk, wg;
    int side;  // -1 left, 1 right, 0 the centre (and the unused lanes 41..63)
};
struct RmargPre {
    Gk41Node g;
    double prior, alp, gam, ginv;
};

// spline_init_ws (GSL cspline_init semantics) by each wave: lane p holds knot (xp, yp) for
// p < n, the knots already in t.s.x and t.s.y.  The rows of the tridiagonal system are formed
// by their lanes at once; the LDL^T recurrences run over lane values read into scalar
// registers, in spline_init_ws's order and with its expressions, so c, and the b_i and d_i
// formed from it, are the same bit for bit.  Wave 0 writes n, linear = 0, c, b and d.
// `whole`: the knots are the whole scalelength grid, whose factorisation (alp, gam and the
// 1 / h) the host formed once with the same expressions (RGrid): what is left is the two
// substitutions, without the 21 dependent divisions.  With the series' read-ahead
// (expint_ei_wave) an evaluation of a 64-dish loop took the small-facet kernel 17.4 us
// instead of 19.9, and the kernel of many items 9.9 instead of 12.1.
// Returns spline_init_ws's status, the same in every lane.
__device__ int spline_build_wave(SplineLds &t, int n, double xp, double yp, bool whole,
                                 const RmargPre &pre)
{
    const int lane = threadIdx.x & 63;
    const bool w0 = threadIdx.x < 64;
    const double x1 = __shfl_down(xp, 1), x2 = __shfl_down(xp, 2);
    const double y1 = __shfl_down(yp, 1), y2 = __shfl_down(yp, 2);
    if (__any(lane + 1 < n && !(xp < x1))) return 1;  // knots strictly increasing
    const int max_index = n - 1, sys = max_index - 1;
    double off = 0., diag = 0., g = 0.;
    const double ginv1 = __shfl_down(pre.ginv, 1);
    if (whole) {
        const double yd_i = y1 - yp;
        const double yd_ip1 = y2 - y1;
        if (lane < sys) g = 3.0 * (yd_ip1 * ginv1 - yd_i * pre.ginv);
    } else if (lane < sys) {
        const double h_i = x1 - xp;
        const double h_ip1 = x2 - x1;
        const double yd_i = y1 - yp;
        const double yd_ip1 = y2 - y1;
        const double g_i = (h_i != 0.0) ? 1.0 / h_i : 0.0;
        const double g_ip1 = (h_ip1 != 0.0) ? 1.0 / h_ip1 : 0.0;
        off = h_ip1;
        diag = 2.0 * (h_ip1 + h_i);
        g = 3.0 * (yd_ip1 * g_ip1 - yd_i * g_i);
    }
    double c = 0.;  // lane p: c_p, with c_0 = c_{n-1} = 0
    int status = 0;
    if (sys == 1) {
        const double c1 = read_lane(g, 0) / read_lane(diag, 0);
        if (lane == 1) c = c1;
    } else if (whole) {
        // every lane takes its row's step again and again from its neighbour's value: lane i
        // has its final value after i steps and keeps it
        const double gam1 = dpp_shift_f64<0x138>(pre.gam);  // lane i: gam_{i-1} (lane 0: 0)
        double z = g;
        for (int i = 1; i < sys; i++) z = g - gam1 * dpp_shift_f64<0x138>(z);
        const double cc = lane < sys ? z / pre.alp : 0.;
        const double gm = lane < sys - 1 ? pre.gam : 0.;
        double xs = cc;
        for (int i = 1; i < sys; i++) xs = cc - gm * dpp_shift_f64<0x130>(xs);
        xs = dpp_shift_f64<0x138>(xs);  // c_{i+1} = x_i
        if (lane >= 1 && lane <= sys) c = xs;
    } else if (sys > 1) {
        // step i: alp_i from gam_{i-1}, the forward substitution's z_i, then gam_i =
        // off_i / alp_i, whose division is the chain's latency; the next step's lane values
        // are read before it
        double alp_l = 0., gam_l = 0., z_l = 0.;  // lane i: alp_i, gam_i, z_i
        double al = read_lane(diag, 0);
        double of = read_lane(off, 0);
        double z = read_lane(g, 0);
        double gm = of / al;
        if (al == 0) status = 1;
        if (lane == 0) {
            alp_l = al;
            gam_l = gm;
            z_l = z;
        }
        double dg = read_lane(diag, 1), gg = read_lane(g, 1), of_next = read_lane(off, 1);
        for (int i = 1; i < sys - 1; i++) {
            al = dg - of * gm;
            z = gg - gm * z;
            of = of_next;
            dg = read_lane(diag, i + 1);
            gg = read_lane(g, i + 1);
            of_next = read_lane(off, i + 1);
            gm = of / al;
            if (al == 0) status = 1;
            if (lane == i) {
                alp_l = al;
                gam_l = gm;
                z_l = z;
            }
        }
        al = dg - of * gm;  // alp_{sys-1}: no gam, and no status check, in spline_init_ws
        z = gg - gm * z;
        if (lane == sys - 1) {
            alp_l = al;
            z_l = z;
        }
        const double cc = lane < sys ? z_l / alp_l : 0.;
        double xs = read_lane(cc, sys - 1);
        if (lane == sys) c = xs;
        for (int i = sys - 2; i >= 0; i--) {
            xs = read_lane(cc, i) - read_lane(gam_l, i) * xs;
            if (lane == i + 1) c = xs;
        }
    }
    const double c1 = __shfl_down(c, 1);
    if (w0) {
        if (lane == 0) {
            t.s.n = n;
            t.s.linear = 0;
        }
        if (lane < n) t.s.c[lane] = c;
        if (lane + 1 < n) {
            const double dx = x1 - xp;
            const double dy = y1 - yp;
            t.b[lane] = (dy / dx) - dx * (c1 + 2.0 * c) / 3.0;
            t.d[lane] = (c1 - c) / (3.0 * dx);
        }
    }
    return status;
}

// Lane j's Gauss-Kronrod-41 node (0..19 left of the centre, 20..39 right, 40 the centre) and
// its Kronrod and Gauss weights, read once per work-group.
__device__ inline Gk41Node gk41_node()
{
    const int lane = threadIdx.x & 63;
    const int k = lane < 20 ? lane : lane - 20;
    Gk41Node g{0., 0., 0., 0};
    if (lane < 41) {
        g.side = lane < 20 ? -1 : (lane < 40 ? 1 : 0);
        g.x = lane < 40 ? kXgk41[k] : 0.;
        g.wk = lane < 40 ? kWgk41[k] : kWgk41[20];
        g.wg = (lane < 40 && (k & 1)) ? kWg41[k >> 1] : 0.;
    }
    return g;
}

__device__ inline void qk41_wave(const SplineLds &sp, const Gk41Node &g, double a, double b,
                                 double *result, double *abserr, double *resabs,
                                 double *resasc)
{
    const int lane = threadIdx.x & 63;
    const double center = 0.5 * (a + b);
    const double half_length = 0.5 * (b - a);
    const double abs_half_length = fabs(half_length);
    double f = 0.;
    if (lane < 41) {
        double x;
        if (g.side < 0)
            x = center - half_length * g.x;
        else if (g.side > 0)
            x = center + half_length * g.x;
        else
            x = center;
        f = spline_exp_lds(sp, x);
    }
    double result_kronrod = wave_sum(g.wk * f);
    const double result_gauss = wave_sum(g.wg * f);
    double result_abs = wave_sum(g.wk * fabs(f));
    const double mean = result_kronrod * 0.5;
    double result_asc = wave_sum(lane < 41 ? g.wk * fabs(f - mean) : 0.);
    const double err = (result_kronrod - result_gauss) * half_length;
    result_kronrod *= half_length;
    result_abs *= abs_half_length;
    result_asc *= abs_half_length;
    *result = result_kronrod;
    *resabs = result_abs;
    *resasc = result_asc;
    *abserr = rescale_error(err, result_abs, result_asc);
}

// qag41_spline's QUADPACK sequence by the work-group.  Each bisection takes two barriers: one
// after the halves' results are exchanged, one after lane 0 has updated the lists (qpsrt
// included) and published the next interval; every thread reads the exchange before the
// second and the lists after it, so no write can overtake a read of the previous bisection.
__device__ int qag41_wave(const SplineLds &sp, const Gk41Node &g, double a, double b,
                          double epsrel, int limit, QagWs &w, double *result)
{
    double result0, abserr0, resabs0, resasc0;
    int roundoff_type1 = 0, roundoff_type2 = 0, error_type = 0;
    const bool writer = threadIdx.x == 0;
    if (writer) {
        w.alist[0] = a;
        w.blist[0] = b;
        w.rlist[0] = 0.0;
        w.elist[0] = 0.0;
        w.order[0] = 0;
        w.level[0] = 0;
    }
    int size = 0, nrmax = 0, imax = 0;
    *result = 0;
    qk41_wave(sp, g, a, b, &result0, &abserr0, &resabs0, &resasc0);
    size = 1;
    if (writer) {
        w.rlist[0] = result0;
        w.elist[0] = abserr0;
    }
    double tolerance = fmax(0., epsrel * fabs(result0));
    const double round_off = 50 * kDblEps * resabs0;
    if (abserr0 <= round_off && abserr0 > tolerance) {
        *result = result0;
        return 14;
    } else if ((abserr0 <= tolerance && abserr0 != resasc0) || abserr0 == 0.0) {
        *result = result0;
        return 0;
    } else if (limit == 1) {
        *result = result0;
        return 11;
    }
    double area = result0, errsum = abserr0;
    int iteration = 1;
    __shared__ double xch[8];
    __shared__ int sh_imax, sh_nrmax;
    __syncthreads();
    do {
        const double a_i = w.alist[imax], b_i = w.blist[imax];
        const double r_i = w.rlist[imax], e_i = w.elist[imax];
        const int lev = w.level[imax];
        const double a1 = a_i, b1 = 0.5 * (a_i + b_i), a2 = b1, b2 = b_i;
        double area1, area2, error1, error2, resasc1, resasc2;  // |f| integrals unused by qag
        // the two halves at once: wave 0 integrates [a1, b1], wave 1 [a2, b2]
        {
            const int wv = threadIdx.x >> 6;
            double r, e, ra, rc;
            qk41_wave(sp, g, wv ? a2 : a1, wv ? b2 : b1, &r, &e, &ra, &rc);
            if ((threadIdx.x & 63) == 0) {
                xch[4 * wv + 0] = r;
                xch[4 * wv + 1] = e;
                xch[4 * wv + 2] = ra;
                xch[4 * wv + 3] = rc;
            }
        }
        __syncthreads();
        area1 = xch[0];
        error1 = xch[1];
        resasc1 = xch[3];
        area2 = xch[4];
        error2 = xch[5];
        resasc2 = xch[7];
        const double area12 = area1 + area2;
        const double error12 = error1 + error2;
        errsum += (error12 - e_i);
        area += area12 - r_i;
        if (resasc1 != error1 && resasc2 != error2) {
            const double delta = r_i - area12;
            if (fabs(delta) <= 1.0e-5 * fabs(area12) && error12 >= 0.99 * e_i) roundoff_type1++;
            if (iteration >= 10 && error12 > e_i) roundoff_type2++;
        }
        tolerance = fmax(0., epsrel * fabs(area));
        if (errsum > tolerance) {
            if (roundoff_type1 >= 6 || roundoff_type2 >= 20) error_type = 2;
            const double tmp = (1 + 100 * kDblEps) * (fabs(a2) + 1000 * kDblMin);
            if (fabs(a1) <= tmp && fabs(b2) <= tmp) error_type = 3;
        }
        size++;
        if (writer) {
            const int i_max = imax, i_new = size - 1;
            const int new_level = lev + 1;
            if (error2 > error1) {
                w.alist[i_max] = a2;
                w.rlist[i_max] = area2;
                w.elist[i_max] = error2;
                w.level[i_max] = new_level;
                w.alist[i_new] = a1;
                w.blist[i_new] = b1;
                w.rlist[i_new] = area1;
                w.elist[i_new] = error1;
                w.level[i_new] = new_level;
            } else {
                w.blist[i_max] = b1;
                w.rlist[i_max] = area1;
                w.elist[i_max] = error1;
                w.level[i_max] = new_level;
                w.alist[i_new] = a2;
                w.blist[i_new] = b2;
                w.rlist[i_new] = area2;
                w.elist[i_new] = error2;
                w.level[i_new] = new_level;
            }
            qpsrt(w, size, limit, nrmax, imax);
            sh_imax = imax;
            sh_nrmax = nrmax;
        }
        __syncthreads();
        imax = sh_imax;
        nrmax = sh_nrmax;
        iteration++;
    } while (iteration < limit && !error_type && errsum > tolerance);
    double sum = 0;
    for (int k = 0; k < size; k++) sum += w.rlist[k];
    *result = sum;
    if (errsum <= tolerance) return 0;
    if (error_type == 2) return 14;
    if (error_type == 3) return 21;
    if (iteration == limit) return 11;
    return 5;
}

__device__ inline RmargPre rmarg_pre(const LikLaunch &a, int slot)
{
    const int lane = threadIdx.x & 63;
    const bool mine = lane < kMaxR;
    RmargPre p;
    p.g = gk41_node();
    p.prior = mine ? a.facets[slot].rprior[lane] : 0.;
    p.alp = mine ? a.rg.alp[lane] : 0.;
    p.gam = mine ? a.rg.gam[lane] : 0.;
    p.ginv = mine ? a.rg.ginv[lane] : 0.;
    return p;
}

// likelihood.c:126-146 with marginalise_posterior_r (marginalise_r.c:81-223) for one item, by
// the two waves of the work-group.  Lane r (1 <= r < numR) of each wave holds L_r[r] in lv; the
// points above kBad go, in r order, to knots 0..num-1 in LDS; ymax is a wave reduction; xmin
// and xmax are the first and the last knot (the extreme abscissae: the reference's start from
// the neighbours of the maximum does not change them, and knots that do not increase are an
// error whatever they are); the QUADPACK lists live in LDS.  fragile: a mixed-precision item
// with a fragile L_r.
__device__ void rmarg_item(const LikLaunch &a, const RmargPre &pre, double lv, bool fragile,
                           int item, SplineLds &sp, double *qd, int *qi)
{
    const int lane = threadIdx.x & 63;
    const int numR = a.rg.numr;
    const bool mine = lane >= 1 && lane < numR;
    const Gk41Node &g = pre.g;
    const bool ok = mine && lv > kBad;
    const double xr = mine ? a.rg.ro[lane] : 0.;
    const double yr = ok ? lv + pre.prior : 0.;
    const uint64_t m = __ballot(ok);
    const int num = __popcll(m);
    int error = 0;
    double L_e;
    if (num > 4) {
        const double ymax = wave_max(ok && yr > -10.0 ? yr : -10.0);
        const int pos = __popcll(m & ((1ull << lane) - 1ull));
        if (threadIdx.x < 64 && ok) {
            sp.s.x[pos] = xr;
            sp.s.y[pos] = yr - ymax;
        }
        __syncthreads();
        const double xp = lane < num ? sp.s.x[lane] : 0.;
        const double yp = lane < num ? sp.s.y[lane] : 0.;
        const double xmin = read_lane(xp, 0), xmax = read_lane(xp, num - 1);
        if (xmax <= xmin ||
            spline_build_wave(sp, num, xp, yp, a.rg.factored && num == numR - 1, pre)) {
            L_e = NAN;
        } else {
            QagWs w;
            w.alist = qd;
            w.blist = qd + kQagLimit;
            w.rlist = qd + 2 * kQagLimit;
            w.elist = qd + 3 * kQagLimit;
            w.order = qi;
            w.level = qi + kQagLimit;
            __syncthreads();
            double sump = 0.;
            int st = qag41_wave(sp, g, xmin, xmax, 1.e-3, kQagLimit, w, &sump);
            if (st) {  // linear interpolation (marginalise_r.c: the retry after a failure)
                __syncthreads();
                if (threadIdx.x == 0) sp.s.linear = 1;
                __syncthreads();
                st = qag41_wave(sp, g, xmin, xmax, 1.e-3, kQagLimit, w, &sump);
            }
            L_e = st ? kBad : log(sump) + ymax;
        }
    } else {
        error = 1;
        L_e = kBad;
    }
    if (L_e == kBad) error = 1;
    if (fragile) error |= kErrFragile;
    if (threadIdx.x == 0) {
        a.Le[item] = L_e;
        a.err[item] = error;
    }
}

__device__ void tile_status(const LikLaunch &a);

// The spline and the QUADPACK interval lists live in LDS (41 KB): lane 0 updates the lists
// and every lane reads them back after each bisection, a round trip through L2 when they
// were in global memory.
__global__ __launch_bounds__(128) void rmarg_kernel(LikLaunch a)
{
    if (blockIdx.x == (unsigned)a.nitems) {  // the status group (tiled engine)
        tile_status(a);
        return;
    }
    __shared__ SplineLds sp;
    __shared__ double qd[kQagDoubles];
    __shared__ int qi[kQagInts];
    const LikItem it = a.items[blockIdx.x];
    const int lane = threadIdx.x & 63;
    const bool mine = lane >= 1 && lane < a.rg.numr;
    // every global read of the item is issued here, the node tables first
    const RmargPre pre = rmarg_pre(a, it.slot);
    const size_t base = (size_t)blockIdx.x * kMaxR;
    const double lv = mine ? a.Lr[base + lane] : kBad;
    bool act = false, frag = false;
    if (a.tasks && mine) {
        act = a.tasks[base + lane].active;
        frag = a.tasks[base + lane].fragile;
    }
    if (__any(act)) return;  // tiled engine: an item with a task still iterating waits
    // the node tables have arrived with the loads above: keep them from being re-read later
    asm volatile("" ::"v"(pre.g.x), "v"(pre.g.wk), "v"(pre.g.wg));
    rmarg_item(a, pre, lv, it.prec == 1 && __any(frag), blockIdx.x, sp, qd, qi);
}

// ------------------------------------------------------------------ likelihood, tiled
// Largest item whose first work-group is <= wg (first work-groups are non-decreasing and
// every item has at least one work-group).
__device__ inline int tile_item(const LikItem *items, int nitems, unsigned wg, int nr_g)
{
    int lo = 0, hi = nitems;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (items[mid].chunk_first * (unsigned)nr_g <= wg)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Work-groups [first, first + nr_g * chunks) of `item`, chunk-major: the nr_g scalelength
// tasks of one chunk are consecutive, so they read the same cells close together in time.
__device__ inline void tile_range(const TileLaunch &t, const LikItem *items, int item,
                                  unsigned *first, unsigned *nch)
{
    if (t.item_chunks) {  // every item of the launch has item_chunks chunks
        *first = (unsigned)item * t.item_chunks * (unsigned)t.nr_g;
        *nch = t.item_chunks;
        return;
    }
    const unsigned c0 = items[item].chunk_first;
    const unsigned c1 = (item + 1 < t.lk.nitems) ? items[item + 1].chunk_first
                                                  : t.nwg / (unsigned)t.nr_g;
    *first = c0 * (unsigned)t.nr_g;
    *nch = c1 - c0;
}

// The item, first work-group and chunk count of logical work-group wg: a division when every
// item of the launch has the same chunk count (one galaxy's points: the serial loop), else
// the search over the items' first chunks.
__device__ inline void tile_locate(const TileLaunch &t, const LikItem *items, unsigned wg,
                                   int *item, unsigned *first, unsigned *nch)
{
    *item = t.item_chunks ? (int)(wg / (t.item_chunks * (unsigned)t.nr_g))
                          : tile_item(items, t.lk.nitems, wg, t.nr_g);
    tile_range(t, items, *item, first, nch);
}

// Work-groups are dispatched to the 8 XCDs round-robin (block b to XCD b % 8) and each XCD
// has its own L2.  The blocks of XCD x walk the logical work-groups x * per ... (x + 1) *
// per - 1 (per = ceil(nwg / 8)), so the tasks of a chunk run on one XCD and share its L2.
// Blocks of a pass: one per logical work-group, or at most `cap` (a multiple of 8).
inline unsigned tile_grid(unsigned nwg, unsigned cap)
{
    const unsigned g = (nwg + kXcds - 1) / kXcds * kXcds;
    return (cap && g > cap) ? cap : g;
}

// Loads through the global address space: the facet arrays are reached through pointers
// read from memory, which the compiler would otherwise address as flat (generic) memory,
// and a flat load also holds the LDS counter every wait has to drain.
#define RL2_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ inline T gload(const T *p, size_t i)
{
    return ((const RL2_GLOBAL T *)p)[i];
}
// HIP's vector structs through the matching builtin vector types (one 16-byte load)
typedef double rl2_d2 __attribute__((ext_vector_type(2)));
typedef float rl2_f4 __attribute__((ext_vector_type(4)));
__device__ inline double2 gload(const double2 *p, size_t i)
{
    const rl2_d2 v = ((const RL2_GLOBAL rl2_d2 *)p)[i];
    return make_double2(v.x, v.y);
}
__device__ inline float4 gload(const float4 *p, size_t i)
{
    const rl2_f4 v = ((const RL2_GLOBAL rl2_f4 *)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}

// Cells per thread whose loads are issued together before any of them is used: a thread
// walks its cells beg + tid, beg + tid + 256, ... in batches of kTileU, so each memory
// round trip serves kTileU cells.  Lanes past the chunk end load cell `beg` with zero data:
// their terms are exactly zero, and every thread adds its cells in increasing order as
// before.
constexpr int kTileU = 4;
// Cells per thread and batch of the paths with two batches in flight (the Newton passes'
// record path, pass 0 on extracted facets; 3 and 4 measured slower).
constexpr int kRecU = 2;

// Chunk sums in FP64.  PASS 0: {S2, value, dx, dy, dxx, dyy, dxy} of the unnormalised
// model at zero offset (likelihood.c:214-236); PASS 1: {value, dx, dy, dxx, dyy, dxy} at
// the offset (xo, yo) (likelihood.c:296-327).
template <int PASS>
__device__ inline void tile_sums64(const FacetDev &F, const LikItem &it, double ro, double xo,
                                   double yo, unsigned beg, unsigned end, double (&s)[7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(ro);
    const double sf = (scale * scale) / (detA * detA);
    const double sw = sf * (4 * kPi * kPi);
    const double a1 = 1. + e1, a2 = 1. - e1;
#pragma unroll
    for (int j = 0; j < 7; j++) s[j] = 0.;
    for (unsigned base = beg + threadIdx.x; base < end; base += kTileU * kTileBS) {
        double uu[kTileU], vv[kTileU], dr[kTileU], di[kTileU], s2[kTileU];
#pragma unroll
        for (int q = 0; q < kTileU; q++) {
            const unsigned i = base + q * kTileBS;
            const bool in = i < end;
            const unsigned k = in ? i : beg;
            uu[q] = gload(F.uu, k);
            vv[q] = gload(F.vv, k);
            const double r_ = gload(F.dre, k), m_ = gload(F.dim, k);
            dr[q] = in ? r_ : 0.;
            di[q] = in ? m_ : 0.;
            s2[q] = PASS == 0 ? gload(F.s2, k) : 1.;
        }
#pragma unroll
        for (int q = 0; q < kTileU; q++) {
            const double k1 = fma(e2, vv[q], a1 * uu[q]);
            const double k2 = fma(a2, vv[q], e2 * uu[q]);
            const double rr = rsqrt_ge1(fma(sw, fma(k1, k1, k2 * k2), 1.));
            const double M = rr * rr * rr;
            const double hr = dr[q] * M;
            const double hi = -di[q] * M;
            const double U = kTwoPi * uu[q], V = kTwoPi * vv[q];
            if (PASS == 0) {
                if (base + q * kTileBS < end) s[0] += M * M / s2[q];
                s[1] += hr;
                s[2] = fma(-hi, U, s[2]);
                s[3] = fma(-hi, V, s[3]);
                const double hU = hr * U;
                s[4] = fma(-hU, U, s[4]);
                s[5] = fma(-hr * V, V, s[5]);
                s[6] = fma(-hU, V, s[6]);
            } else {
                // phase xo U + yo V = 2 pi (xo u + yo v): evaluated in revolutions
                double sn, cs;
                sincos_rev64(fma(xo, uu[q], yo * vv[q]), sn, cs);
                const double re = fma(hr, cs, -hi * sn);
                const double im = fma(hr, sn, hi * cs);
                s[0] += re;
                s[1] = fma(-im, U, s[1]);
                s[2] = fma(-im, V, s[2]);
                const double rU = re * U;
                s[3] = fma(-rU, U, s[3]);
                s[4] = fma(-re * V, V, s[4]);
                s[5] = fma(-rU, V, s[5]);
            }
        }
    }
}

// PASS 0 sums of tile_sums64 on a facet with grid structure: the cell centres from the
// LDS copy of ctr (sC) by cell id, so a cell costs 28 bytes of vector memory instead of 40,
// and M^2 / sigma^2 as M^2 times the packed 1 / sigma^2 (one rounding apart from the
// quotient; the division sequence was a fifth of the pass's instructions).
template <int U>
__device__ inline void tile_sums64_p0_grid(const FacetDev &F, const LikItem &it, double ro,
                                           const double *sC, unsigned beg, unsigned end,
                                           double (&s)[7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(ro);
    const double sf = (scale * scale) / (detA * detA);
    const double sw = sf * (4 * kPi * kPi);
    const double a1 = 1. + e1, a2 = 1. - e1;
#pragma unroll
    for (int j = 0; j < 7; j++) s[j] = 0.;
    for (unsigned base = beg + threadIdx.x; base < end; base += U * kTileBS) {
        uint32_t c[U];
        double dr[U], di[U], s2[U];
#pragma unroll
        for (int q = 0; q < U; q++) {
            const unsigned i = base + q * kTileBS;
            const unsigned k = i < end ? i : F.n;  // past the end: the zero pad cell
            c[q] = gload(F.cid, k);
            dr[q] = gload(F.dre, k);
            di[q] = gload(F.dim, k);
            s2[q] = gload(F.invs2_64, k);  // 1 / sigma^2
        }
#pragma unroll
        for (int q = 0; q < U; q++) {
            const double uu = sC[c[q] & 0xffffu], vv = sC[c[q] >> 16];
            const double k1 = fma(e2, vv, a1 * uu);
            const double k2 = fma(a2, vv, e2 * uu);
            const double rr = rsqrt_ge1(fma(sw, fma(k1, k1, k2 * k2), 1.));
            const double M = rr * rr * rr;
            const double hr = dr[q] * M;
            const double hi = -di[q] * M;
            // sums over u, v: the 2 pi and 4 pi^2 factors are applied to the totals below
            s[0] = fma(M * M, s2[q], s[0]);
            s[1] += hr;
            s[2] = fma(-hi, uu, s[2]);
            s[3] = fma(-hi, vv, s[3]);
            const double hU = hr * uu;
            s[4] = fma(-hU, uu, s[4]);
            s[5] = fma(-hr * vv, vv, s[5]);
            s[6] = fma(-hU, vv, s[6]);
        }
    }
    s[2] *= kTwoPi;
    s[3] *= kTwoPi;
    constexpr double kTwoPi2 = kTwoPi * kTwoPi;
    s[4] *= kTwoPi2;
    s[5] *= kTwoPi2;
    s[6] *= kTwoPi2;
}

// tile_sums64_p0_grid's sums with two batches of kRecU cells per thread in flight: the next
// batch's loads are issued before the current batch is summed, the visibility pair comes from
// the packed copy dc, and `stage` (the centres into sC, ending with a barrier) runs after the
// first batch's loads are issued.  A thread's cells, and so its sums, are those of
// tile_sums64_p0_grid in the same order (past the end: the zero pad cell, which adds zeros).
// NT scalelength tasks of the same item and chunk at once (ro[t], s[t]): the cell's loads,
// centres and the shape terms k1, k2 and k1^2 + k2^2 are shared, the rest is each task's own,
// with the expressions of the one-task form, so every task's sums are the same bit for bit.
template <int NT, class Stage>
__device__ inline void tile_sums64_p0_db(const FacetDev &F, const LikItem &it,
                                         const double (&ro)[NT], const double *sC,
                                         const Stage &stage, unsigned beg, unsigned end,
                                         double (&s)[NT][7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    double sw[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const double scale = arcs2rad_scale(ro[t]);
        const double sf = (scale * scale) / (detA * detA);
        sw[t] = sf * (4 * kPi * kPi);
    }
    const double a1 = 1. + e1, a2 = 1. - e1;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < 7; j++) s[t][j] = 0.;
    const uint32_t *cid = F.cid;
    const double2 *dc = F.dc;
    const double *w2 = F.invs2_64;
    const unsigned pad = F.n;
    struct Cells {
        uint32_t c[kRecU];
        double dr[kRecU], di[kRecU], s2[kRecU];
    };
    auto fetch = [&](Cells &b, unsigned base) {
#pragma unroll
        for (int q = 0; q < kRecU; q++) {
            const unsigned i = base + q * kTileBS;
            const unsigned k = i < end ? i : pad;
            b.c[q] = gload(cid, k);
            const double2 d = gload(dc, k);
            b.dr[q] = d.x;
            b.di[q] = d.y;
            b.s2[q] = gload(w2, k);
        }
    };
    auto eval = [&](const Cells &b) {
#pragma unroll
        for (int q = 0; q < kRecU; q++) {
            const double uu = sC[b.c[q] & 0xffffu], vv = sC[b.c[q] >> 16];
            const double k1 = fma(e2, vv, a1 * uu);
            const double k2 = fma(a2, vv, e2 * uu);
            const double kk = fma(k1, k1, k2 * k2);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const double rr = rsqrt_ge1(fma(sw[t], kk, 1.));
                const double M = rr * rr * rr;
                const double hr = b.dr[q] * M;
                const double hi = -b.di[q] * M;
                s[t][0] = fma(M * M, b.s2[q], s[t][0]);
                s[t][1] += hr;
                s[t][2] = fma(-hi, uu, s[t][2]);
                s[t][3] = fma(-hi, vv, s[t][3]);
                const double hU = hr * uu;
                s[t][4] = fma(-hU, uu, s[t][4]);
                s[t][5] = fma(-hr * vv, vv, s[t][5]);
                s[t][6] = fma(-hU, vv, s[t][6]);
            }
        }
    };
    constexpr unsigned S = kRecU * kTileBS;
    Cells A, B;
    fetch(A, beg + threadIdx.x);
    stage();
#pragma unroll
    for (int q = 0; q < kRecU; q++)
        asm volatile("" : "+v"(A.c[q]), "+v"(A.dr[q]), "+v"(A.di[q]), "+v"(A.s2[q]));
    for (unsigned base = beg + threadIdx.x; base < end; base += 2 * S) {
        fetch(B, base + S);
        __builtin_amdgcn_sched_barrier(0);
        eval(A);
        if (base + S >= end) break;
        fetch(A, base + 2 * S);
        __builtin_amdgcn_sched_barrier(0);
        eval(B);
    }
    constexpr double kTwoPi2 = kTwoPi * kTwoPi;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        s[t][2] *= kTwoPi;
        s[t][3] *= kTwoPi;
        s[t][4] *= kTwoPi2;
        s[t][5] *= kTwoPi2;
        s[t][6] *= kTwoPi2;
    }
}

// PASS 1 sums of tile_sums64 on a facet with grid structure.  The Newton phase is
// separable on the grid, 2 pi (xo u + yo v) with u = ctr[column], v = ctr[row], so
// e^{i phase} is the product of the task's column entry X[column] = e^{2 pi i xo u} and row
// entry Y[row] = e^{2 pi i yo v}, computed once per pass (lik_step_kernel) instead of a
// sin/cos per cell.  The cell centres come from ctr, bit-identical to uu / vv.  The work-group
// copies X, ctr and (YL) Y to LDS first (sX, sC, sY): per cell only the cell id and data then
// go through the vector memory pipeline, which otherwise carried 68 bytes per cell and task.
// Without YL the row entry is a global load, nearly uniform across a wave.
// One batch of cells of the table path: cell ids and data.
constexpr int kTabU = 2;
struct TabCells {
    uint32_t c[kTabU];
    double dr[kTabU], di[kTabU];
};

// `stage` fills sX, sC and (YL) sY and ends with a barrier; it runs after the first cells'
// loads are issued, so their round trip overlaps it.  It returns false (the same in every
// thread) when the work-group has nothing to sum; the function then returns false too.
template <bool YL, class Stage>
__device__ inline bool tile_sums64_tab(const FacetDev &F, const LikItem &it, double ro,
                                       const Stage &stage, const double2 *Yg, double2 *sX,
                                       double2 *sY, double *sC, unsigned beg, unsigned end,
                                       double (&s)[7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(ro);
    const double sf = (scale * scale) / (detA * detA);
    const double sw = sf * (4 * kPi * kPi);
    const double a1 = 1. + e1, a2 = 1. - e1;
#pragma unroll
    for (int j = 0; j < 7; j++) s[j] = 0.;
    // The facet fields in registers (the scheduling barriers below would otherwise make the
    // compiler reload them from the descriptor every iteration).  Lanes past the end of the
    // chunk read the zero pad cell after the facet's last one, so the loads are
    // unconditional and no lane masks its data.
    const uint32_t *cid = F.cid;
    const double *dre = F.dre, *dim = F.dim;
    const unsigned pad = F.n;
    auto fetch = [&](TabCells &b, unsigned base) {
#pragma unroll
        for (int q = 0; q < kTabU; q++) {
            const unsigned i = base + q * kTileBS;
            const unsigned k = i < end ? i : pad;
            b.c[q] = gload(cid, k);
            b.dr[q] = gload(dre, k);
            b.di[q] = gload(dim, k);
        }
    };
    auto eval = [&](const TabCells &b) {
        double uu[kTabU], vv[kTabU];
        double2 x[kTabU], y[kTabU];
#pragma unroll
        for (int q = 0; q < kTabU; q++) {
            const unsigned ci = b.c[q] & 0xffffu, cj = b.c[q] >> 16;
            uu[q] = sC[ci];
            vv[q] = sC[cj];
            x[q] = sX[ci];
            y[q] = YL ? sY[cj] : gload(Yg, cj);
        }
#pragma unroll
        for (int q = 0; q < kTabU; q++) {
            const double k1 = fma(e2, vv[q], a1 * uu[q]);
            const double k2 = fma(a2, vv[q], e2 * uu[q]);
            const double rr = rsqrt_ge1(fma(sw, fma(k1, k1, k2 * k2), 1.));
            const double M = rr * rr * rr;
            const double hr = b.dr[q] * M;
            const double hi = -b.di[q] * M;
            const double cs = fma(x[q].x, y[q].x, -(x[q].y * y[q].y));
            const double sn = fma(x[q].y, y[q].x, x[q].x * y[q].y);
            const double re = fma(hr, cs, -hi * sn);
            const double im = fma(hr, sn, hi * cs);
            // the gradient and Hessian sums over u, v; their 2 pi and 4 pi^2 factors are
            // applied once to the thread's totals instead of to every cell's U = 2 pi u
            s[0] += re;
            s[1] = fma(-im, uu[q], s[1]);
            s[2] = fma(-im, vv[q], s[2]);
            const double rU = re * uu[q];
            s[3] = fma(-rU, uu[q], s[3]);
            s[4] = fma(-re * vv[q], vv[q], s[4]);
            s[5] = fma(-rU, vv[q], s[5]);
        }
    };
    // Software-pipelined over two register sets: the loads of the next batch are issued
    // before the current batch is evaluated, so their latency overlaps its arithmetic.  A
    // set is loaded only after its previous batch has been used, so the loop needs no
    // register copies (a copy of a just-issued load waits for it at once), and the
    // scheduling barriers keep the loads above the arithmetic.  The first batch passes
    // through an empty asm so that the compiler does not fold the loop-carried set back
    // into loads at the point of use.  Cells are still added in increasing order.
    constexpr unsigned S = kTabU * kTileBS;
    TabCells A, B;
    // the first cells are requested before the tables are staged in LDS, so the two
    // memory round trips at the start of the work-group overlap
    fetch(A, beg + threadIdx.x);
    if (!stage()) return false;
#pragma unroll
    for (int q = 0; q < kTabU; q++) asm volatile("" : "+v"(A.c[q]), "+v"(A.dr[q]), "+v"(A.di[q]));
    for (unsigned base = beg + threadIdx.x; base < end; base += 2 * S) {
        fetch(B, base + S);
        __builtin_amdgcn_sched_barrier(0);
        eval(A);
        if (base + S >= end) break;
        fetch(A, base + 2 * S);
        __builtin_amdgcn_sched_barrier(0);
        eval(B);
    }
    s[1] *= kTwoPi;
    s[2] *= kTwoPi;
    constexpr double kTwoPi2 = kTwoPi * kTwoPi;
    s[3] *= kTwoPi2;
    s[4] *= kTwoPi2;
    s[5] *= kTwoPi2;
    return true;
}

// The Newton-pass sums of tile_sums64_tab from LDS records: grid index k's record at byte
// k * kRecBytes holds {X[k], Y[k], ctr[k]} as five doubles (8-byte aligned: read in pairs),
// and a cell's packed loff gives both its records' offsets, so per cell the vector memory
// carries loff and the packed {D_re, D_im}, and the LDS addresses need no arithmetic
// beyond unpacking.  The arithmetic and its order are tile_sums64_tab's.
struct RecEntry {
    double xr, xi, yr, yi, c;
};
// The cell centres as the records hold them (RecEntry::c), indexed like the centre array.
struct RecCtr {
    const RecEntry *rec;
    __device__ double operator[](unsigned k) const { return rec[k].c; }
};
static_assert(sizeof(RecEntry) == kRecBytes, "record layout");
struct RecCells {
    uint32_t o[kRecU];
    double dr[kRecU], di[kRecU];
};
template <class Stage>
__device__ inline bool tile_sums64_rec(unsigned pad, const uint32_t *loff, const double2 *dc,
                                       const LikItem &it, double ro,
                                       const Stage &stage, const char *rec, unsigned beg,
                                       unsigned end, double (&s)[7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(ro);
    const double sf = (scale * scale) / (detA * detA);
    const double sw = sf * (4 * kPi * kPi);
    const double a1 = 1. + e1, a2 = 1. - e1;
#pragma unroll
    for (int j = 0; j < 7; j++) s[j] = 0.;
    auto fetch = [&](RecCells &b, unsigned base) {
#pragma unroll
        for (int q = 0; q < kRecU; q++) {
            const unsigned i = base + q * kTileBS;
            const unsigned k = i < end ? i : pad;
            b.o[q] = gload(loff, k);
            const double2 d = gload(dc, k);
            b.dr[q] = d.x;
            b.di[q] = d.y;
        }
    };
    auto eval = [&](const RecCells &b) {
        double uu[kRecU], vv[kRecU];
        double2 x[kRecU], y[kRecU];
#pragma unroll
        for (int q = 0; q < kRecU; q++) {
            const RecEntry &col = *reinterpret_cast<const RecEntry *>(rec + (b.o[q] & 0xffffu));
            const RecEntry &row = *reinterpret_cast<const RecEntry *>(rec + (b.o[q] >> 16));
            uu[q] = col.c;
            vv[q] = row.c;
            x[q] = make_double2(col.xr, col.xi);
            y[q] = make_double2(row.yr, row.yi);
        }
#pragma unroll
        for (int q = 0; q < kRecU; q++) {
            const double k1 = fma(e2, vv[q], a1 * uu[q]);
            const double k2 = fma(a2, vv[q], e2 * uu[q]);
            const double rr = rsqrt_ge1(fma(sw, fma(k1, k1, k2 * k2), 1.));
            const double M = rr * rr * rr;
            const double hr = b.dr[q] * M;
            const double hi = -b.di[q] * M;
            const double cs = fma(x[q].x, y[q].x, -(x[q].y * y[q].y));
            const double sn = fma(x[q].y, y[q].x, x[q].x * y[q].y);
            const double re = fma(hr, cs, -hi * sn);
            const double im = fma(hr, sn, hi * cs);
            s[0] += re;
            s[1] = fma(-im, uu[q], s[1]);
            s[2] = fma(-im, vv[q], s[2]);
            const double rU = re * uu[q];
            s[3] = fma(-rU, uu[q], s[3]);
            s[4] = fma(-re * vv[q], vv[q], s[4]);
            s[5] = fma(-rU, vv[q], s[5]);
        }
    };
    constexpr unsigned S = kRecU * kTileBS;
    RecCells A, B;
    fetch(A, beg + threadIdx.x);
    if (!stage()) return false;
#pragma unroll
    for (int q = 0; q < kRecU; q++) asm volatile("" : "+v"(A.o[q]), "+v"(A.dr[q]), "+v"(A.di[q]));
    for (unsigned base = beg + threadIdx.x; base < end; base += 2 * S) {
        fetch(B, base + S);
        __builtin_amdgcn_sched_barrier(0);
        eval(A);
        if (base + S >= end) break;
        fetch(A, base + 2 * S);
        __builtin_amdgcn_sched_barrier(0);
        eval(B);
    }
    s[1] *= kTwoPi;
    s[2] *= kTwoPi;
    constexpr double kTwoPi2 = kTwoPi * kTwoPi;
    s[3] *= kTwoPi2;
    s[4] *= kTwoPi2;
    s[5] *= kTwoPi2;
    return true;
}

// The same sums from the FP32 facet copy: model and terms in FP32, the per-thread FP32
// partials added into FP64 every kFlush cells; the Newton phase formed and reduced in
// FP64 revolutions.
template <int PASS>
__device__ inline void tile_sums32(const FacetDev &F, const LikItem &it, double ro, double xo,
                                   double yo, unsigned beg, unsigned end, double (&s)[7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(ro);
    const double sf = (scale * scale) / (detA * detA);
    const float sw = (float)(sf * (4 * kPi * kPi));
    const float a1 = (float)(1. + e1), a2 = (float)(1. - e1), fe2 = (float)e2;
    const float tp = 6.28318530717958648f;
#pragma unroll
    for (int j = 0; j < 7; j++) s[j] = 0.;
    for (unsigned base = beg + threadIdx.x; base < end; base += kFlush * kTileBS) {
        float f[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const unsigned stop = min(end, base + kFlush * kTileBS);
#pragma unroll 2
        for (unsigned i = base; i < stop; i += kTileBS) {
            const float4 p = gload(F.pk, i);
            const float k1 = fmaf(fe2, p.y, a1 * p.x);
            const float k2 = fmaf(a2, p.y, fe2 * p.x);
            const float rr = rsqrtf(fmaf(sw, fmaf(k1, k1, k2 * k2), 1.f));
            const float M = rr * rr * rr;
            const float hr = p.z * M;
            const float hi = -p.w * M;
            const float U = tp * p.x, V = tp * p.y;
            if (PASS == 0) {
                f[0] = fmaf(M * M, gload(F.invs2, i), f[0]);
                f[1] += hr;
                f[2] = fmaf(-hi, U, f[2]);
                f[3] = fmaf(-hi, V, f[3]);
                const float hU = hr * U;
                f[4] = fmaf(-hU, U, f[4]);
                f[5] = fmaf(-hr * V, V, f[5]);
                f[6] = fmaf(-hU, V, f[6]);
            } else {
                float sn, cs;
                sincos_rev(fma(xo, (double)p.x, yo * (double)p.y), sn, cs);
                const float re = fmaf(hr, cs, -hi * sn);
                const float im = fmaf(hr, sn, hi * cs);
                f[0] += re;
                f[1] = fmaf(-im, U, f[1]);
                f[2] = fmaf(-im, V, f[2]);
                const float rU = re * U;
                f[3] = fmaf(-rU, U, f[3]);
                f[4] = fmaf(-re * V, V, f[4]);
                f[5] = fmaf(-rU, V, f[5]);
            }
        }
#pragma unroll
        for (int j = 0; j < 7; j++) s[j] += (double)f[j];
    }
}

// The Newton loop of likelihood.c:284-350 one step at a time: the task's state T advances
// by the step from the sums v (PASS 0: the zero-offset sums, which also start the state);
// returns 1 when the task has finished, with ho and the normalised determinant for L_r.
template <int PASS>
__device__ int newton_update(TileTask &T, const double (&v)[7], double *ho_out,
                             double *det_out)
{
    double value, dx, dy, dxx, dyy, dxy;
    if (PASS == 0) {
        T.S2 = v[0];
        value = v[1];
        dx = v[2];
        dy = v[3];
        dxx = v[4];
        dyy = v[5];
        dxy = v[6];
        T.xo = 0.;
        T.yo = 0.;
        T.norm = 1.;
        T.iter = 0;
        T.fragile = 0;
    } else {
        value = v[0];
        dx = v[1];
        dy = v[2];
        dxx = v[3];
        dyy = v[4];
        dxy = v[5];
    }
    const double det = dxx * dyy - dxy * dxy;
    if (det > 0 && T.norm > 1.e-7 && T.iter < 50) {
        const double incx = (dx * dyy - dy * dxy) / det;
        const double incy = (dy * dxx - dx * dxy) / det;
        T.xo -= incx;
        T.yo -= incy;
        T.iter += 1;
        T.norm = sqrt(incx * incx + incy * incy);
        T.active = 1;
        return 0;
    }
    T.active = 0;
    const double S2 = T.S2;
    // branches an FP32 sum could decide differently: the determinant sign, the Newton
    // step cap, the position-marginalisation cut x <= Delta (likelihood.c:395)
    const double ho = value / sqrt(S2);
    const double scale = fabs(dxx * dyy) + dxy * dxy;
    const double B = ho * ho * 0.5, Delta = 0.5 * 5.991;
    T.fragile = (fabs(det) <= 1e-5 * scale) || T.iter >= 50 ||
                fabs(B - Delta) <= 1e-4 * fabs(B) || !isfinite(det);
    *ho_out = ho;
    *det_out = det / S2;
    return 1;
}

// newton_update on the task's state in memory, writing L_r when the task finishes (the
// step kernel of the two-kernel passes).
// The state is read from T and written to To (the same task in another buffer when the
// passes keep two generations of state; T itself otherwise).  Called by a whole wave with the
// same sums in every lane; lane 0 writes the state.
template <int PASS>
__device__ int tile_step(const LikLaunch &a, const TileTask *T, TileTask *To, int item, int r,
                         const double (&v)[7], double *xo, double *yo)
{
    TileTask S = *T;
    double ho, det;
    const int done = newton_update<PASS>(S, v, &ho, &det);
    if ((threadIdx.x & 63) == 0) *To = S;
    if (done) finish_lr(a, item, r, ho, det, S.iter);
    *xo = S.xo;
    *yo = S.yo;
    return done;
}

// A task's chunk sums of one pass added by one wave in a fixed order, with the totals in every
// lane: the chunks are paired by bit 0 of their number (mod 64), then bit 1, and so on.  Lane l
// reads value l % 8 of chunks 8 i + l / 8 (and those 64, 128, ... further, added first) for
// each block i of eight chunks; a block adds up over its lanes, then the blocks by pairs.
// read(i, c): the lane's sum over the chunks c, c + 64, ... below nch of block i.
template <class Read>
__device__ inline void task_totals(unsigned nch, const Read &read, double (&v)[7])
{
    const int lane = threadIdx.x & 63;
    double t[8];
#pragma unroll
    for (unsigned i = 0; i < 8; i++)
        t[i] = 8 * i < nch ? wave_sum_by8(read(i, 8 * i + (lane >> 3))) : 0.;
    const double s = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
#pragma unroll
    for (int j = 0; j < 7; j++) v[j] = read_lane(s, j);
}
// P0 is the task's first chunk; chunk c follows at c * nr * 8.
__device__ inline void task_sums(const double *P0, unsigned nch, int nr, int lane,
                                 double (&v)[7])
{
    task_totals(nch,
                [&](unsigned, unsigned c) {
                    double t = 0.;
                    for (; c < nch; c += 64) t += P0[(size_t)c * nr * 8 + (lane & 7)];
                    return t;
                },
                v);
}

// Newton phase tables e^{2 pi i o ctr[k]} (o = xo for the columns, yo for the rows) by runs
// of kTabRun grid indices.  The cell centres are evenly spaced, ctr[k] = (k + 0.5) inc - len
// (evaluate_uv_grid.c:127-128), so ctr[run * kTabRun + j] - ctr[run * kTabRun] equals
// ctr[j] - ctr[0] to within a few ulp of len: entry k is the product of the run's first
// entry E[k / kTabRun] (sincos_rev64) and W[k % kTabRun] = e^{2 pi i o (ctr[j] - ctr[0])}, one
// sin/cos per run and per run offset instead of one per entry.  The step kernel and the
// fused passes build their tables this same way, so both give the same entries.
constexpr unsigned kTabRun = 16;
template <unsigned NRUN>
struct TabRot {
    double2 ex[NRUN], ey[NRUN], wx[kTabRun], wy[kTabRun];
};
__device__ inline double2 cis_rev(double t)
{
    double sn, cs;
    sincos_rev64(t, sn, cs);
    return make_double2(cs, sn);
}
__device__ inline double2 tab_entry(const double2 &e, const double2 &w)
{
    return make_double2(fma(e.x, w.x, -(e.y * w.y)), fma(e.y, w.x, e.x * w.y));
}
// The runs' first entries (columns: every run of the gf columns; rows: runs yb0..yb1 and,
// with y0, run 0) and both W tables, spread over the block's threads; the caller
// synchronises before reading R.  ctr(k): the cell centre k, from global memory or from a
// copy in LDS.
template <unsigned NRUN, class Ctr>
__device__ inline void tab_rot_stage(TabRot<NRUN> &R, const Ctr &ctr, unsigned gf, double xo,
                                     double yo, unsigned yb0, unsigned yb1, bool y0)
{
    const unsigned nb = (gf + kTabRun - 1) / kTabRun;
    const unsigned ny = yb1 - yb0 + 1 + (y0 ? 1u : 0u);
    const unsigned nw = min(gf, kTabRun);
    const double c0 = ctr[0];
    static_assert(sizeof(TabRot<NRUN>) == (2 * NRUN + 2 * kTabRun) * sizeof(double2),
                  "ex, ey, wx, wy contiguous");
    double2 *E = reinterpret_cast<double2 *>(&R);  // ex, ey, wx, wy in that order
    for (unsigned q = threadIdx.x; q < nb + ny + 2 * nw; q += blockDim.x) {
        // the entry's centre index, factor and slot by selects, then one centre read and one
        // sin/cos whatever the kind of entry: with them in branches, a wave holding several
        // kinds ran each branch's read and sin/cos one after the other
        const bool isx = q < nb, isy = !isx && q < nb + ny;
        const unsigned b = q - nb <= yb1 - yb0 ? yb0 + (q - nb) : 0u;  // a row run (isy)
        const unsigned w = q - nb - ny;                                  // < 2 nw (W entries)
        const unsigned j = w < nw ? w : w - nw;
        const unsigned ci = isx ? q * kTabRun : (isy ? b * kTabRun : j);
        const double o = isx ? xo : (isy ? yo : (w < nw ? xo : yo));
        const unsigned slot =
            isx ? q : (isy ? NRUN + b : 2 * NRUN + (w < nw ? 0u : kTabRun) + j);
        const double c = ctr[ci];
        const double run = o * c, off = o * (c - c0);  // a run's first entry; a W entry
        E[slot] = cis_rev(isx || isy ? run : off);
    }
}
template <unsigned NRUN>
__device__ inline double2 tab_x(const TabRot<NRUN> &R, unsigned k)
{
    return tab_entry(R.ex[k / kTabRun], R.wx[k % kTabRun]);
}
template <unsigned NRUN>
__device__ inline double2 tab_y(const TabRot<NRUN> &R, unsigned k)
{
    return tab_entry(R.ey[k / kTabRun], R.wy[k % kTabRun]);
}

// The chunk sums of a tile work-group into P[0..7]: each wave's totals, then thread j adds the
// waves' value j in wave order.
__device__ inline void tile_reduce(double (&v)[7], double *lds, double *P)
{
    constexpr int NW = kTileBS / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double w[8] = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], 0.};
    const double s = wave_sum8(w);
    if (lane < 8) lds[wave * 8 + lane] = s;
    __syncthreads();
    if (threadIdx.x < 8) {
        double t = 0.;
#pragma unroll
        for (int q = 0; q < NW; q++) t += lds[q * 8 + threadIdx.x];
        P[threadIdx.x] = t;
    }
    __syncthreads();  // lds is reused by the block's next logical work-group
}

template <int PASS, int KIND>
__device__ inline void tile_chunk(const TileLaunch &t, unsigned wg, double *red);

// Waves per SIMD the tile kernels are compiled for.  The generic kernel carries every path
// (the FP32 sums and the per-cell sin/cos among them) in 128 VGPRs; the grid kernel only
// the FP64 paths of extracted facets (pass 0 with the cell centres in LDS, Newton passes
// from the phase tables), which fit a smaller register budget, so more waves stay resident
// to cover the memory latency.
constexpr int kTileWaves = 4;
#ifndef RL2_TILE_GRID_WAVES
#define RL2_TILE_GRID_WAVES 4
#endif
constexpr int kTileGridWaves = RL2_TILE_GRID_WAVES;

// A block takes the logical work-groups q, q + nbx, q + 2 nbx, ... of its XCD's eighth of
// the logical order (q = block / 8, nbx = blocks per XCD): with one block per logical
// work-group that is exactly one, and a launch capped at the resident block count walks
// the whole pass without further dispatches.
template <int PASS, int KIND>
__global__ __launch_bounds__(kTileBS, KIND ? kTileGridWaves : kTileWaves) void lik_tile_kernel(
    TileLaunch t)
{
    __shared__ double red[(kTileBS / 64) * 8];
    if (PASS == 0 && blockIdx.x == 0 && threadIdx.x < t.n_inl)
        t.items_w[threadIdx.x] = t.inl[threadIdx.x];
    const unsigned per = (t.nwg + kXcds - 1) / kXcds;
    const unsigned nbx = gridDim.x / kXcds;
    for (unsigned j = blockIdx.x / kXcds; j < per; j += nbx) {
        const unsigned wg = (blockIdx.x % kXcds) * per + j;
        if (wg >= t.nwg) break;
        tile_chunk<PASS, KIND>(t, wg, red);
    }
}

// KIND 0: any items (the generic kernel).  KIND 1 and 2 (the grid kernels): every item of
// the launch is an FP64 item on an extracted facet with phase tables, which the host checks
// when it picks the kernel; KIND 2 when the items travel in the kernel arguments.
template <int PASS, int KIND>
__device__ inline void tile_chunk(const TileLaunch &t, unsigned wg, double *red)
{
    constexpr bool GRID = KIND != 0;
    const LikLaunch &a = t.lk;
    // KIND 2: the items from the kernel arguments (scalar loads that stay in the scalar
    // cache instead of a chain of dependent vector loads for the search).  Pass 0 reads them
    // there whenever they travel there: its block 0 is what stores them to a.items.
    const LikItem *items =
        KIND == 2 ? t.inl : ((PASS == 0 && t.n_inl) ? t.inl : a.items);
    int item;
    unsigned first, nch;
    tile_locate(t, items, wg, &item, &first, &nch);
    const unsigned local = wg - first;
    const unsigned chunk = local / (unsigned)t.nr_g;
    const int r = (int)(local - chunk * (unsigned)t.nr_g) + t.r_lo;
    const TileTask *T = t.tasks + (size_t)item * kMaxR + r;
    if (PASS == 1 && !T->active) return;  // finished task: the whole work-group moves on
    const LikItem it = items[item];
    const unsigned beg = chunk * it.chunk_cells;
    double s[7];
    if constexpr (GRID) {
        auto grid_sums = [&](const FacetDev &F) {
            const unsigned end = min(F.n, beg + it.chunk_cells);
            extern __shared__ double2 tab_lds[];
            if (PASS == 1) {
                // t.tab_lds_facet * (16 + 8) bytes, + 16 with the rows: X, ctr, Y
                const unsigned gf = F.grid_facet;
                const double2 *X = t.tab + it.tab_first + (size_t)(r - 1) * 2 * gf;
                const double2 *Y = X + gf;
                double2 *sX = tab_lds;
                double *sC = reinterpret_cast<double *>(tab_lds + t.tab_lds_facet);
                double2 *sY = reinterpret_cast<double2 *>(sC + t.tab_lds_facet);
                const bool yl = t.tab_y_lds;
                auto copy = [&]() {  // the step kernel's tables and the cell centres
                    const double *ctr = F.ctr;
                    for (unsigned k = threadIdx.x; k < gf; k += kTileBS) {
                        sX[k] = gload(X, k);
                        sC[k] = gload(ctr, k);
                        if (yl) sY[k] = gload(Y, k);
                    }
                    __syncthreads();
                    return true;
                };
                if (yl)
                    tile_sums64_tab<true>(F, it, a.rg.ro[r], copy, Y, sX, sY, sC, beg, end, s);
                else
                    tile_sums64_tab<false>(F, it, a.rg.ro[r], copy, Y, sX, sY, sC, beg, end, s);
            } else {
                double *sC = reinterpret_cast<double *>(tab_lds);  // tab_lds_facet * 8 bytes
                auto stage = [&]() {
                    for (unsigned k = threadIdx.x; k < F.grid_facet; k += kTileBS)
                        sC[k] = gload(F.ctr, k);
                    __syncthreads();
                };
                const double ro1[1] = {a.rg.ro[r]};
                tile_sums64_p0_db<1>(F, it, ro1, sC, stage, beg, end,
                                     reinterpret_cast<double(&)[1][7]>(s));
            }
        };
        grid_sums(a.facets[it.slot]);
    } else {
        const FacetDev &F = a.facets[it.slot];
        const unsigned end = min(F.n, beg + it.chunk_cells);
        if (PASS == 1 && it.prec == 0 && t.tab && F.cid) {
            extern __shared__ double2 tab_lds[];
            const unsigned gf = F.grid_facet;
            const double2 *X = t.tab + it.tab_first + (size_t)(r - 1) * 2 * gf;
            const double2 *Y = X + gf;
            double2 *sX = tab_lds;
            double *sC = reinterpret_cast<double *>(tab_lds + t.tab_lds_facet);
            double2 *sY = reinterpret_cast<double2 *>(sC + t.tab_lds_facet);
            const bool yl = t.tab_y_lds;
            auto copy = [&]() {
                const double *ctr = F.ctr;
                for (unsigned k = threadIdx.x; k < gf; k += kTileBS) {
                    sX[k] = gload(X, k);
                    sC[k] = gload(ctr, k);
                    if (yl) sY[k] = gload(Y, k);
                }
                __syncthreads();
                return true;
            };
            if (yl)
                tile_sums64_tab<true>(F, it, a.rg.ro[r], copy, Y, sX, sY, sC, beg, end, s);
            else
                tile_sums64_tab<false>(F, it, a.rg.ro[r], copy, Y, sX, sY, sC, beg, end, s);
        } else if (PASS == 0 && it.prec == 0 && F.cid && F.grid_facet <= t.tab_lds_facet) {
            extern __shared__ double2 tab_lds[];  // t.tab_lds_facet * 8 bytes: ctr
            double *sC = reinterpret_cast<double *>(tab_lds);
            for (unsigned k = threadIdx.x; k < F.grid_facet; k += kTileBS)
                sC[k] = gload(F.ctr, k);
            __syncthreads();
            tile_sums64_p0_grid<kTileU>(F, it, a.rg.ro[r], sC, beg, end, s);
        } else if (it.prec == 0)
            tile_sums64<PASS>(F, it, a.rg.ro[r], PASS == 1 ? T->xo : 0.,
                              PASS == 1 ? T->yo : 0., beg, end, s);
        else
            tile_sums32<PASS>(F, it, a.rg.ro[r], PASS == 1 ? T->xo : 0.,
                              PASS == 1 ? T->yo : 0., beg, end, s);
    }
    tile_reduce(s, red, t.partials + (size_t)wg * 8);
}

// One work-group per (item, r) task.  Wave 0 adds the task's chunk sums in a fixed order and
// takes the Newton step or ends the task; when the task goes on over a grid facet in FP64, the whole group (16 waves, so each lane
// writes at most 3 entries of the 2 * facet) then writes its phase tables for the next pass.
constexpr int kStepBS = 1024;
template <int PASS>
__global__ __launch_bounds__(kStepBS) void lik_step_kernel(TileLaunch t)
{
    __shared__ int s_go;
    __shared__ double s_off[2];
    const LikLaunch &a = t.lk;
    const int nr = t.nr_g;
    const unsigned k = blockIdx.x;
    const int item = (int)(k / nr), r = (int)(k % nr) + t.r_lo;
    TileTask *T = t.tasks + (size_t)item * kMaxR + r;
    TileTask *To = (t.tasks_out ? t.tasks_out : t.tasks) + (size_t)item * kMaxR + r;
    // the item and its facet fields are requested by every wave at once, so their latency
    // overlaps the reduction instead of following the barrier
    const LikItem it = a.items[item];
    const FacetDev &F = a.facets[it.slot];
    const uint32_t *fcid = F.cid;
    const double *fctr = F.ctr;
    const unsigned gf = F.grid_facet;
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        int go = 0;
        if (PASS == 0 || T->active) {  // read by the whole wave before lane 0 updates it
            unsigned first, nch;
            tile_range(t, a.items, item, &first, &nch);
            double v[7];
            task_sums(t.partials + (size_t)(first + (unsigned)(r - t.r_lo)) * 8, nch, nr, lane,
                      v);
            double xo, yo;
            go = !tile_step<PASS>(a, T, To, item, r, v, &xo, &yo);
            if (lane == 0) {
                s_off[0] = xo;
                s_off[1] = yo;
            }
        } else if (lane == 0 && To != T) {
            *To = *T;  // a finished task keeps its state in the other generation too
        }
        if (lane == 0) s_go = go;
    }
    __syncthreads();
    if (!s_go || !t.tab) return;
    if (it.prec != 0 || !fcid) return;
    double2 *X = t.tab + it.tab_first + (size_t)(r - 1) * 2 * gf;
    // every column and every row (gf <= 1706: the host's LDS limit for the column tables)
    __shared__ TabRot<128> R;
    const unsigned nb = (gf + kTabRun - 1) / kTabRun;
    tab_rot_stage(R, fctr, gf, s_off[0], s_off[1], 0u, nb - 1, false);
    __syncthreads();
    for (unsigned q = threadIdx.x; q < 2 * gf; q += blockDim.x)
        X[q] = q < gf ? tab_x(R, q) : tab_y(R, q - gf);
}


// status[0] = tasks still iterating, status[1] = largest Newton step count,
// *flops = sum over tasks of n (37 + 25 N_it) (model + normalisation 19, zero-offset sums
// 18, 25 per Newton pass; transcendentals, sqrt and division counted as one).  Run by the
// first wave of one extra work-group of the r-marginalisation launch.
__device__ void tile_status(const LikLaunch &a)
{
    if (threadIdx.x >= 64) return;
    const int nr = a.rg.numr - 1;
    const unsigned ntask = (unsigned)a.nitems * nr;
    unsigned c = 0, m = 0;
    double f = 0.;
    for (unsigned k = threadIdx.x; k < ntask; k += 64) {
        const int item = (int)(k / nr);
        const TileTask &T = a.tasks[(size_t)item * kMaxR + k % nr + 1];
        c += T.active ? 1u : 0u;
        m = max(m, (unsigned)T.iter);
        f += (double)a.facets[a.items[item].slot].n * (37. + 25. * T.iter);
    }
    for (int off = 32; off >= 1; off >>= 1) {
        c += __shfl_xor(c, off);
        m = max(m, (unsigned)__shfl_xor((int)m, off));
        f += __shfl_xor(f, off);
    }
    if (threadIdx.x == 0) {
        a.status[0] = c;
        a.status[1] = m;
        *a.flops = f;
    }
}

// ------------------------------------------------------------------ Newton passes, fused
// What a fused pass's work-group reads of its task before anything else, so that these
// loads are in flight with the facet's and the cells': the task's state S (the same address
// in every thread: scalar loads) and wave 0's share of the previous pass's chunk sums of the
// task (task_sums' lanes, when nch <= 8 kPreChunks; task_sums reads them itself otherwise).
constexpr unsigned kPreChunks = 4;
struct FusedPre {
    TileTask S;
    double p[kPreChunks];
};

__device__ __attribute__((always_inline)) inline FusedPre fused_pre(const TileLaunch &t,
                                                                    unsigned first,
                                                                    unsigned nch, int item,
                                                                    int r)
{
    FusedPre f;
    f.S = t.tasks[(size_t)item * kMaxR + r];
    const unsigned lane = threadIdx.x;
    const bool read = t.mode != 2 && nch <= 8 * kPreChunks && lane < 64;
    const double *P = t.part_in + (size_t)(first + (unsigned)(r - t.r_lo)) * 8 + (lane & 7);
#pragma unroll
    for (unsigned k = 0; k < kPreChunks; k++) {
        const unsigned c = (lane >> 3) + 8 * k;
        f.p[k] = 0.;
        if (read && 8 * k < nch && c < nch) f.p[k] = P[(size_t)c * t.nr_g * 8];
    }
    return f;
}

// The step a fused pass's work-group takes before its sums (wave 0; the caller
// synchronises), for a task that is still iterating (fused_idle has dealt with the others):
// the task's chunk sums of the previous pass added in chunk order, the Newton step, the
// state stored by the task's chunk-0 work-group (to the other generation) with L_r when the
// task ends; *go and off[2] receive whether the task goes on and its new offset.
__device__ __attribute__((always_inline)) inline void fused_step(const TileLaunch &t, unsigned first,
                                                                 unsigned nch,
                                  unsigned chunk, int item, int r, const FusedPre &pre,
                                  int *go_out, double *off)
{
    if (threadIdx.x >= 64) return;
    const LikLaunch &a = t.lk;
    const size_t ti = (size_t)item * kMaxR + r;
    const int lane = threadIdx.x;
    int go = 0;
    double xo = 0., yo = 0.;
    if (t.mode == 2) {
        go = pre.S.active;
        xo = pre.S.xo;
        yo = pre.S.yo;
    } else {
        double v[7];
        if (nch <= 8 * kPreChunks) {  // task_sums' arithmetic on the chunk sums read at the start
            task_totals(nch,
                        [&](unsigned i, unsigned) {
                            double p = i < kPreChunks ? pre.p[i < kPreChunks ? i : 0] : 0.;
                            asm volatile("" : "+v"(p));  // consumed here, not at the load's issue
                            return p;
                        },
                        v);
        } else {
            task_sums(t.part_in + (size_t)(first + (unsigned)(r - t.r_lo)) * 8, nch, t.nr_g,
                      lane, v);
        }
        // every lane takes the step from the same totals: the end of a task is the wave's
        TileTask S = t.mode == 0 ? TileTask{} : pre.S;
        double ho, det;
        const int done = t.mode == 0 ? newton_update<0>(S, v, &ho, &det)
                                     : newton_update<1>(S, v, &ho, &det);
        if (chunk == 0) {
            if (lane == 0) t.tasks_out[ti] = S;
            if (done) finish_lr(a, item, r, ho, det, S.iter);
        }
        go = !done;
        xo = S.xo;
        yo = S.yo;
    }
    if (lane == 0) {
        *go_out = go;
        off[0] = xo;
        off[1] = yo;
    }
}

// Whether a fused pass's work-group has a task that ended in an earlier pass (mode 1), in
// which case the task's chunk-0 work-group keeps its state in both generations.  Every wave
// holds the flag (read with scalar loads, whose wait does not include the cells' vector
// loads in flight), so an idle work-group leaves without a barrier, which would wait for
// those loads.
__device__ inline bool fused_idle(const TileLaunch &t, unsigned chunk, int item, int r,
                                  const FusedPre &pre)
{
    if (t.mode != 1 || pre.S.active) return false;
    if (chunk == 0 && threadIdx.x == 63) t.tasks_out[(size_t)item * kMaxR + r] = pre.S;
    return true;
}

// One Newton pass with the previous pass's step folded in, so that a pass is one launch
// instead of two.  Each work-group first adds its task's chunk sums of the previous pass
// (wave 0, in the step kernel's order) and takes the Newton step itself, so every
// work-group of a task holds the same state bit for bit.  The task's chunk-0 work-group
// stores that state to the other generation of the task buffer (the rest of the pass still
// reads this one) and writes L_r when the task ends.  The work-group then evaluates its own
// phase tables in LDS with the step kernel's arithmetic: the column table over the facet's
// width, the row table over the rows its chunk spans (cells are in row-major order) and row
// 0, which the zero pad cell reads.  t.mode: 0 the first step, from the pass-0 sums; 1 a
// Newton step from the previous pass's sums; 2 resume from the state the step kernel left.
template <int KIND>
__global__ __launch_bounds__(kTileBS, kTileGridWaves) void lik_fused_kernel(TileLaunch t)
{
    __shared__ double red[(kTileBS / 64) * 8];
    __shared__ int s_go;
    __shared__ double s_off[2];
    // one block per logical work-group, in the XCD-aware order of lik_tile_kernel
    const unsigned per = (t.nwg + kXcds - 1) / kXcds;
    const unsigned wg = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (wg >= t.nwg) return;
    const LikLaunch &a = t.lk;
    const LikItem *items = KIND == 2 ? t.inl : a.items;
    int item;
    unsigned first, nch;
    tile_locate(t, items, wg, &item, &first, &nch);
    const unsigned local = wg - first;
    const unsigned chunk = local / (unsigned)t.nr_g;
    const int r = (int)(local - chunk * (unsigned)t.nr_g) + t.r_lo;
    const FusedPre pre = fused_pre(t, first, nch, item, r);
    const LikItem it = items[item];
    const FacetDev &F = a.facets[it.slot];
    const unsigned fn = F.n;
    const unsigned gf = F.grid_facet;  // <= 1024: the host checks the LDS tables fit
    const uint32_t *cid = F.cid, *loff = F.loff;
    const double *ctr = F.ctr;
    const double2 *dc = F.dc;
    // the facet's fields arrive with the task's state: one wait for both, before the
    // cells' loads are issued
    asm volatile("" ::"s"(fn), "s"(gf), "s"(cid), "s"(loff), "s"(ctr), "s"(dc));
    const unsigned beg = chunk * it.chunk_cells;
    const unsigned end = min(fn, beg + it.chunk_cells);
    extern __shared__ double2 tab_lds[];  // t.tab_lds_facet records of kRecBytes
    RecEntry *rec = reinterpret_cast<RecEntry *>(tab_lds);
    // Runs after the first cells' loads are issued (inside tile_sums64_rec): the cell
    // centres this thread's records need are requested too, then wave 0 adds the previous
    // pass's chunk sums and takes the step while those loads are in flight.
    __shared__ TabRot<1024 / kTabRun> R;  // gf <= 1024
    auto make = [&]() -> bool {
        if (fused_idle(t, chunk, item, r, pre)) return false;
        constexpr int NC = 1024 / kTileBS;
        double c[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) {  // loads without branches: one count of them to wait on
            const unsigned k = threadIdx.x + j * kTileBS;
            const double v = gload(ctr, k < gf ? k : 0u);
            c[j] = k < gf ? v : 0.;
        }
        uint32_t id_lo = end > beg ? gload(cid, beg) : 0u;
        uint32_t id_hi = end > beg ? gload(cid, end - 1) : 0u;
        fused_step(t, first, nch, chunk, item, r, pre, &s_go, s_off);
        // the records' centres do not depend on the step: stored while wave 0 takes it, and
        // the tables read their runs' centres from them
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const unsigned k = threadIdx.x + j * kTileBS;
            if (k < gf) rec[k].c = c[j];
        }
        __syncthreads();
        if (!s_go) return false;
        // the chunk's first and last cell ids are waited for only here: a wait for them
        // before the step would also wait for every cell and centre load issued before them
        asm volatile("" : "+v"(id_lo), "+v"(id_hi));
        const unsigned row_lo = __builtin_amdgcn_readfirstlane(id_lo >> 16);
        const unsigned row_hi = __builtin_amdgcn_readfirstlane(id_hi >> 16);
        // the column runs, the runs of the rows the chunk spans (cells are in row-major
        // order) and run 0 (row 0: the zero pad cell's), then the entries
        const unsigned yb0 = row_lo / kTabRun, yb1 = row_hi / kTabRun;
        tab_rot_stage(R, RecCtr{rec}, gf, s_off[0], s_off[1], yb0, yb1, yb0 > 0);
        __syncthreads();
        // the column entries: every run and W value read before any is used
        double2 ex[NC], wx[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const unsigned k = threadIdx.x + j * kTileBS;
            const unsigned kk = k < gf ? k : 0u;
            ex[j] = R.ex[kk / kTabRun];
            wx[j] = R.wx[kk % kTabRun];
        }
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const unsigned k = threadIdx.x + j * kTileBS;
            if (k < gf) {
                const double2 x = tab_entry(ex[j], wx[j]);
                rec[k].xr = x.x;
                rec[k].xi = x.y;
            }
        }
        const unsigned span = row_hi - row_lo + 1;
        for (unsigned q = threadIdx.x; q < span + (row_lo > 0 ? 1u : 0u); q += kTileBS) {
            const unsigned k = q < span ? row_lo + q : 0u;
            const double2 y = tab_y(R, k);
            rec[k].yr = y.x;
            rec[k].yi = y.y;
        }
        __syncthreads();
        return true;
    };
    double s[7];
    if (tile_sums64_rec(fn, loff, dc, it, a.rg.ro[r], make, reinterpret_cast<const char *>(rec),
                        beg, end, s))
        tile_reduce(s, red, t.partials + (size_t)wg * 8);
}

// ------------------------------------------------------------------ one launch per evaluation
// tile_reduce, with the chunk's sums published to the other work-groups of the launch: the
// stores are made at agent scope, wave 0 (which issued them) waits until they have
// completed, and only then counts the chunk as done on the task's counter.  A reader that
// sees the count loads the sums at agent scope too.  Every sum lives at its own address for
// the whole launch (one slice per pass), so no reader can hold an older copy of it.
__device__ inline void tile_reduce_publish(double (&v)[7], double *lds, double *P, unsigned *cnt)
{
    constexpr int NW = kTileBS / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double w[8] = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], 0.};
    const double s = wave_sum8(w);
    if (lane < 8) lds[wave * 8 + lane] = s;
    __syncthreads();
    if (threadIdx.x < 64) {
        if (threadIdx.x < 8) {
            double t = 0.;
#pragma unroll
            for (int q = 0; q < NW; q++) t += lds[q * 8 + threadIdx.x];
            __hip_atomic_store(P + threadIdx.x, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (threadIdx.x == 0)
            __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();  // lds is reused by the next chunk
}

// A task's chunk sums of one pass as task_sums, loaded at agent scope (published by
// tile_reduce_publish in other work-groups of the launch).
__device__ inline void task_sums_published(const double *P0, unsigned nch, int nr, int lane,
                                           double (&v)[7])
{
    task_totals(nch,
                [&](unsigned, unsigned c) {
                    double t = 0.;
                    for (; c < nch; c += 64)
                        t += __hip_atomic_load(P0 + (size_t)c * nr * 8 + (lane & 7),
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    return t;
                },
                v);
}

// One block's share of an evaluation: a task, and the run of its chunks the block sums.
struct PersistTask {
    int item, r;
    unsigned c0, c1;       // chunks [c0, c1) of the task
    unsigned nch;          // the task's chunk count
    unsigned first;        // its item's first work-group index (chunk-major layout)
    int active;
    int pad;
    TileTask S;            // the block's copy of the task's Newton state
};

// Every Newton pass of one likelihood evaluation, to convergence, in one cooperative launch
// after the pass-0 launch, so that no Newton pass pays a launch, a ramp and a tail.  Work layout:
// XCD x (blocks b with b % 8 == x) owns chunks [x nc / 8, (x + 1) nc / 8) of every task
// (nc: the task's chunk count), so the tasks that read the same cells share that XCD's L2;
// within the XCD the (task, chunk) pairs are listed task by task and each block takes an
// equal contiguous run of the list, so a block holds one or a few tasks and takes their
// Newton steps and builds their phase tables once per pass.  The chunks, their sums and
// the steps are those of the fused passes, bit for bit.
// Between passes a task's chunk sums of pass q >= 1 are complete when its counter reaches
// q nc (pass 0's are complete at launch).  A block waits on that count only for its own task's previous pass, and it
// has finished all its work of every earlier pass, so a waiting block always depends on
// blocks that are running or done: with every block resident (cooperative launch) the
// waits end.  Each wait is bounded all the same (p.spin_limit polls): a block that gives
// up leaves its tasks marked active, which the host reports as an error.

template <int KIND>
__global__ __launch_bounds__(kTileBS, kTileGridWaves) void lik_persist_kernel(PersistLaunch p)
{
    __shared__ double red[(kTileBS / 64) * 8];
    __shared__ PersistTask s_task[kPersistTasks];
    __shared__ int s_ntask, s_go, s_fail;
    __shared__ double s_off[2];
    __shared__ TabRot<1024 / kTabRun> R;
    extern __shared__ double2 tab_lds[];  // t.tab_lds_facet records
    RecEntry *rec = reinterpret_cast<RecEntry *>(tab_lds);
    const TileLaunch &t = p.t;
    const LikLaunch &a = t.lk;
    const LikItem *items = KIND == 2 ? t.inl : a.items;
    const int nr = t.nr_g;
    const unsigned x = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
    // items that travel in the arguments are stored for the r-marginalisation
    if (KIND == 2 && blockIdx.x == 0 && threadIdx.x < t.n_inl)
        t.items_w[threadIdx.x] = t.inl[threadIdx.x];
    if (threadIdx.x == 0) {
        // the XCD's list: item by item, task by task, the task's chunks in the XCD's eighth
        auto chunks = [&](int i) {
            const unsigned c1 = i + 1 < a.nitems ? items[i + 1].chunk_first : t.nwg / nr;
            return c1 - items[i].chunk_first;
        };
        unsigned long long W = 0;
        for (int i = 0; i < a.nitems; i++) {
            const unsigned nc = chunks(i);
            W += (unsigned long long)nr * ((x + 1) * nc / kXcds - x * nc / kXcds);
        }
        const unsigned long long q0 = j * W / p.nbx, q1 = (j + 1) * W / p.nbx;
        int nt = 0;
        unsigned long long P = 0;
        for (int i = 0; i < a.nitems && P < q1 && nt >= 0; i++) {
            const unsigned nc = chunks(i);
            const unsigned lo = x * nc / kXcds, m = (x + 1) * nc / kXcds - lo;
            for (int r = 1; r <= nr && m; r++, P += m) {
                if (P + m <= q0 || P >= q1) continue;
                if (nt == kPersistTasks) {
                    nt = -1;
                    break;
                }
                PersistTask &k = s_task[nt++];
                k.item = i;
                k.r = r;
                k.c0 = lo + (unsigned)(q0 > P ? q0 - P : 0);
                k.c1 = lo + (unsigned)(q1 < P + m ? q1 - P : m);
                k.nch = nc;
                k.first = items[i].chunk_first * (unsigned)nr;
                k.active = 1;
            }
        }
        s_ntask = nt;
        s_fail = 0;
    }
    __syncthreads();
    const int ntask = s_ntask;  // < 0: more tasks than a block holds (the host prevents it)
    // the owner of a task's chunk 0 publishes its state: active until it finishes
    for (int k = 0; k < ntask; k++)
        if (threadIdx.x == 0 && s_task[k].c0 == 0)
            p.t.tasks[(size_t)s_task[k].item * kMaxR + s_task[k].r].active = 1;
    // pass 0's sums are in slice 0 already (the pass-0 launch before this one, stream-ordered);
    // passes 1 .. kPersistPasses - 1 sum; the last iteration only takes the final step
    for (int pass = 1; pass <= kPersistPasses && ntask > 0; pass++) {
        bool any = false;
        for (int k = 0; k < ntask; k++) {
            PersistTask &K = s_task[k];
            if (!K.active) continue;  // uniform: read after a barrier
            const LikItem it = items[K.item];
            const FacetDev &F = a.facets[it.slot];
            const unsigned gf = F.grid_facet;
            const size_t ti = (size_t)K.item * kMaxR + K.r;
            const double ro = a.rg.ro[K.r];
            {
                // the previous pass's sums of this task, then its Newton step
                if (threadIdx.x == 0 && pass > 1) {
                    const unsigned want = (unsigned)(pass - 1) * K.nch;
                    unsigned spins = 0;
                    while (__hip_atomic_load(p.cnt + ti, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT) < want) {
                        if (++spins > p.spin_limit) {
                            s_fail = 1;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                __syncthreads();
                if (s_fail) return;  // the task stays marked active: the host reports it
                if (threadIdx.x < 64) {
                    const int lane = threadIdx.x;
                    double v[7];
                    task_sums_published(p.part + ((size_t)(pass - 1) * t.nwg + K.first +
                                                  (unsigned)(K.r - 1)) * 8,
                                        K.nch, nr, lane, v);
                    TileTask S = pass == 1 ? TileTask{} : K.S;
                    double ho, det;
                    const int done = pass == 1 ? newton_update<0>(S, v, &ho, &det)
                                               : newton_update<1>(S, v, &ho, &det);
                    if (lane == 0) {
                        K.S = S;
                        K.active = !done;
                        if (done && K.c0 == 0) p.t.tasks[ti] = S;
                        s_off[0] = S.xo;
                        s_off[1] = S.yo;
                    }
                    if (done && K.c0 == 0) finish_lr(a, K.item, K.r, ho, det, S.iter);
                }
                __syncthreads();
                if (!K.active) continue;
                // phase tables: every column, the rows this block's cells span, row 0
                const unsigned beg = K.c0 * it.chunk_cells;
                const unsigned end = min(F.n, K.c1 * it.chunk_cells);
                const uint32_t *cid = F.cid;
                const unsigned row_lo = end > beg ? gload(cid, beg) >> 16 : 0u;
                const unsigned row_hi = end > beg ? gload(cid, end - 1) >> 16 : 0u;
                const unsigned yb0 = row_lo / kTabRun, yb1 = row_hi / kTabRun;
                tab_rot_stage(R, F.ctr, gf, s_off[0], s_off[1], yb0, yb1, yb0 > 0);
                __syncthreads();
                for (unsigned q = threadIdx.x; q < gf; q += kTileBS) {
                    const double2 xx = tab_x(R, q);
                    rec[q].xr = xx.x;
                    rec[q].xi = xx.y;
                    rec[q].c = gload(F.ctr, q);
                }
                const unsigned span = row_hi - row_lo + 1;
                for (unsigned q = threadIdx.x; q < span + (row_lo > 0 ? 1u : 0u); q += kTileBS) {
                    const unsigned kk = q < span ? row_lo + q : 0u;
                    const double2 y = tab_y(R, kk);
                    rec[kk].yr = y.x;
                    rec[kk].yi = y.y;
                }
                __syncthreads();
            }
            any = true;
            for (unsigned c = K.c0; c < K.c1; c++) {
                const unsigned beg = c * it.chunk_cells;
                const unsigned end = min(F.n, beg + it.chunk_cells);
                double s[7];
                auto none = []() { return true; };  // the records are already staged
                tile_sums64_rec(F.n, F.loff, F.dc, it, ro, none,
                                reinterpret_cast<const char *>(rec), beg, end, s);
                tile_reduce_publish(
                    s, red, p.part + ((size_t)pass * t.nwg + K.first + c * nr + (K.r - 1)) * 8,
                    p.cnt + ti);
            }
            __syncthreads();  // the records are restaged for the next task
        }
        if (!any) break;
    }
}

// ------------------------------------------------------------------ small facets: one launch
// The whole Newton search of one (item, r) task in one work-group, for facets of at most
// kTaskChunks chunks of kTileMinCells cells with records (up to kRecFacet columns).  Such a
// pass is latency: a launch per pass took 5 to 8 us, of which the cells are a few hundred
// nanoseconds; here a pass is three barriers, and what is left of it is the chain of sums,
// step, tables and cells.  Each group of 256 threads holds the cells of its NC chunks in
// registers: D M (the model M does not depend on the offset) and the record offsets, so a
// Newton pass reads only the records in LDS.  The chunks, a thread's cells and their order,
// the chunk sums, the step and the table entries are those of pass 0 and the fused passes, so
// every L_r is the same bit for bit by either route.
// G groups of 256 threads; a task has at most G * NC chunks (chunk c: group c % G).
// KIND 2 (up to kInlItems items, in the arguments): the work-group that ends an item's last
// task also integrates over the scalelength (rmarg_item), so an evaluation is one launch.
// With more items its lists (40 KB of LDS) would cost the task work-groups their residency,
// and a launch of their own is a small part of the evaluation.
// Measured against the passes: one point on 138 cells 64.1 -> 46.5 us, the loop over 24
// galaxies of 175 to 2111 cells 38.5 -> 26.3 ms, in batches of 16 (48 galaxies) 18.4 -> 15.1
// ms (32 us, 17 and 9 ms with the shorter chains, the integral folded in and the results polled
// for).  On 6,582 cells 1, 4 and 24 points took 69, 71 and 102 us by the passes and 60, 60 and
// 96 here; from 8,192 cells on (twice the cells in registers, which spill) 71, 77 and 128
// against 75, 76 and 139, so kTaskChunks is 4.
template <int KIND, int G, int NC>
__global__ __launch_bounds__(kTileBS *G, NC == 1 ? 4 : 2) void lik_task_kernel(TileLaunch t)
{
    constexpr int BS = kTileBS * G, Q = kTileMinCells / kTileBS, W = kTileBS / 64;
    constexpr int NJ = 8;
    __shared__ double red[G * NC][W][NJ];
    __shared__ TabRot<kRecFacet / kTabRun> R;
    extern __shared__ double2 tab_lds[];  // t.tab_lds_facet records
    RecEntry *rec = reinterpret_cast<RecEntry *>(tab_lds);
    const char *recb = reinterpret_cast<const char *>(tab_lds);
    const LikLaunch &a = t.lk;
    const int item = (int)(blockIdx.x / (unsigned)t.nr_g);
    const int r = (int)(blockIdx.x - (unsigned)item * (unsigned)t.nr_g) + t.r_lo;
    const LikItem it = (KIND == 2 ? t.inl : a.items)[item];
    const FacetDev &F = a.facets[it.slot];
    const unsigned n = F.n, gf = F.grid_facet;
    const uint32_t *loff = F.loff;
    const double2 *dc = F.dc;
    const double *w2 = F.invs2_64, *ctr = F.ctr;
    const unsigned nch = max(1u, (n + kTileMinCells - 1) / kTileMinCells);
    const int g = threadIdx.x / kTileBS, lt = threadIdx.x % kTileBS;
    const int lane = threadIdx.x & 63, wave = (threadIdx.x / 64) % W;
    // rows of 256 cells of the group's chunk k that hold any cell (uniform over the group)
    auto rows = [&](int k) {
        const unsigned beg = (unsigned)(g + k * G) * kTileMinCells;
        return beg < n ? min((unsigned)Q, (n - beg + kTileBS - 1) / kTileBS) : 0u;
    };
    // the thread's cells: offsets and data, then D M (past the end: the zero pad cell n)
    uint32_t o[NC][Q];
    double hr[NC][Q], hi[NC][Q], s2[NC][Q];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const unsigned nq = rows(k);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            if ((unsigned)q >= nq) break;
            const unsigned i =
                min(n, (unsigned)(g + k * G) * kTileMinCells + q * kTileBS + (unsigned)lt);
            o[k][q] = gload(loff, i);
            const double2 d = gload(dc, i);
            hr[k][q] = d.x;
            hi[k][q] = d.y;
            s2[k][q] = gload(w2, i);
        }
    }
    for (unsigned k = threadIdx.x; k < gf; k += BS) rec[k].c = gload(ctr, k);
    __syncthreads();
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(a.rg.ro[r]);
    const double sf = (scale * scale) / (detA * detA);
    const double sw = sf * (4 * kPi * kPi);
    const double a1 = 1. + e1, a2 = 1. - e1;
    constexpr double kTwoPi2 = kTwoPi * kTwoPi;
    // a chunk's sums of this wave
    auto put = [&](int k, double (&s)[NJ]) {
        const double x = wave_sum8(s);
        if (lane < 8) red[g + k * G][wave][lane] = x;
    };
#pragma unroll
    for (int k = 0; k < NC; k++) {  // pass 0: tile_sums64_p0_db's terms
        double s[NJ] = {};
        const unsigned nq = rows(k);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            if ((unsigned)q >= nq) break;
            const double uu = reinterpret_cast<const RecEntry *>(recb + (o[k][q] & 0xffffu))->c;
            const double vv = reinterpret_cast<const RecEntry *>(recb + (o[k][q] >> 16))->c;
            const double k1 = fma(e2, vv, a1 * uu);
            const double k2 = fma(a2, vv, e2 * uu);
            const double rr = rsqrt_ge1(fma(sw, fma(k1, k1, k2 * k2), 1.));
            const double M = rr * rr * rr;
            const double dr = hr[k][q], di = hi[k][q];
            hr[k][q] = dr * M;
            hi[k][q] = -di * M;
            s[0] = fma(M * M, s2[k][q], s[0]);
            s[1] += hr[k][q];
            s[2] = fma(-hi[k][q], uu, s[2]);
            s[3] = fma(-hi[k][q], vv, s[3]);
            const double hU = hr[k][q] * uu;
            s[4] = fma(-hU, uu, s[4]);
            s[5] = fma(-hr[k][q] * vv, vv, s[5]);
            s[6] = fma(-hU, vv, s[6]);
        }
        s[2] *= kTwoPi;
        s[3] *= kTwoPi;
        s[4] *= kTwoPi2;
        s[5] *= kTwoPi2;
        s[6] *= kTwoPi2;
        put(k, s);
    }
    TileTask S = {};
    double ho, det;
    for (int pass = 0;; pass++) {
        __syncthreads();
        // every wave adds the task's chunk sums (tile_reduce's order over the waves, then
        // task_sums' over the chunks) and takes the step
        static_assert(G * NC <= 8, "one block of chunks");
        double v[7];
        task_totals(min(nch, (unsigned)(G * NC)),
                    [&](unsigned, unsigned c) {
                        double p = 0.;
                        if (c < nch && c < G * NC) {
#pragma unroll
                            for (int w = 0; w < W; w++) p += red[c][w][lane & 7];
                        }
                        return p;
                    },
                    v);
        const int done = pass == 0 ? newton_update<0>(S, v, &ho, &det)
                                   : newton_update<1>(S, v, &ho, &det);
        if (done) break;  // the same in every wave
        // the state in scalar registers: the loop's vector registers hold the cells
        S.xo = read_lane(S.xo, 0);
        S.yo = read_lane(S.yo, 0);
        S.norm = read_lane(S.norm, 0);
        S.S2 = read_lane(S.S2, 0);
        S.iter = __builtin_amdgcn_readfirstlane(S.iter);
        tab_rot_stage(R, RecCtr{rec}, gf, S.xo, S.yo, 0u, (gf + kTabRun - 1) / kTabRun - 1, false);
        __syncthreads();
        for (unsigned q = threadIdx.x; q < 2 * gf; q += BS) {
            const unsigned k = q < gf ? q : q - gf;
            const double2 e = q < gf ? tab_x(R, k) : tab_y(R, k);
            double *d = q < gf ? &rec[k].xr : &rec[k].yr;
            d[0] = e.x;
            d[1] = e.y;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NC; k++) {  // tile_sums64_rec's terms
            double s[NJ] = {};
            const unsigned nq = rows(k);
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if ((unsigned)q >= nq) break;
                const RecEntry &col =
                    *reinterpret_cast<const RecEntry *>(recb + (o[k][q] & 0xffffu));
                const RecEntry &row = *reinterpret_cast<const RecEntry *>(recb + (o[k][q] >> 16));
                const double uu = col.c, vv = row.c;
                const double cs = fma(col.xr, row.yr, -(col.xi * row.yi));
                const double sn = fma(col.xi, row.yr, col.xr * row.yi);
                const double re = fma(hr[k][q], cs, -hi[k][q] * sn);
                const double im = fma(hr[k][q], sn, hi[k][q] * cs);
                s[0] += re;
                s[1] = fma(-im, uu, s[1]);
                s[2] = fma(-im, vv, s[2]);
                const double rU = re * uu;
                s[3] = fma(-rU, uu, s[3]);
                s[4] = fma(-re * vv, vv, s[4]);
                s[5] = fma(-rU, vv, s[5]);
            }
            s[1] *= kTwoPi;
            s[2] *= kTwoPi;
            s[3] *= kTwoPi2;
            s[4] *= kTwoPi2;
            s[5] *= kTwoPi2;
            put(k, s);
        }
    }
    if constexpr (KIND != 2) {
        if (threadIdx.x < 64) finish_lr(a, item, r, ho, det, S.iter);
    } else {
        __shared__ SplineLds sp;
        __shared__ bool s_last;
        if (threadIdx.x >= 128) return;
        // in flight while the task ends: what the integral reads besides the L_r
        const RmargPre pre = rmarg_pre(a, it.slot);
        asm volatile("" ::"v"(pre.g.x), "v"(pre.g.wk), "v"(pre.g.wg));
        if (threadIdx.x < 64) finish_lr(a, item, r, ho, det, S.iter);
        if (threadIdx.x == 0) {
            // lane 0 stored L_r at agent scope: the store has completed before the count (the
            // fences of a release and an acquire write back and drop the XCD's whole L2)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const unsigned k = __hip_atomic_fetch_add(t.arrived + item, 1u, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
            s_last = k + 1 == (unsigned)t.nr_g;
            if (s_last)  // zero again for the next launch
                __hip_atomic_store(t.arrived + item, 0u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!s_last) return;
        const double lv = lane >= 1 && lane < a.rg.numr
                              ? __hip_atomic_load(a.Lr + (size_t)item * kMaxR + lane,
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                              : kBad;
        double *qd = reinterpret_cast<double *>(tab_lds);  // the records are done with
        rmarg_item(a, pre, lv, false, item, sp, qd, reinterpret_cast<int *>(qd + kQagDoubles));
    }
}

template <int KIND>
static void launch_task_kind(hipStream_t s, const TileLaunch &t, unsigned chunks)
{
    const unsigned g = (unsigned)t.lk.nitems * (unsigned)t.nr_g;
    unsigned lds = t.tab_lds_facet * kRecBytes;
    if (KIND == 2) lds = std::max(lds, (unsigned)(kQagDoubles * 8 + kQagInts * 4));
    if (chunks <= 1)
        lik_task_kernel<KIND, 1, 1><<<g, kTileBS, lds, s>>>(t);
    else if (chunks <= 2)
        lik_task_kernel<KIND, 2, 1><<<g, 2 * kTileBS, lds, s>>>(t);
    else
        lik_task_kernel<KIND, 2, 2><<<g, 2 * kTileBS, lds, s>>>(t);
}

void launch_lik_task(hipStream_t s, const TileLaunch &t, unsigned chunks)
{
    if (t.grid == 2)
        launch_task_kind<2>(s, t, chunks);
    else
        launch_task_kind<1>(s, t, chunks);
}

// Largest block count of a cooperative persistent launch with `lds` bytes of dynamic LDS
// (0: the kernel cannot run).
unsigned persist_capacity(unsigned lds, int kind)
{
    static std::map<std::pair<unsigned, int>, unsigned> cache;
    const auto key = std::make_pair(lds, kind);
    auto f = cache.find(key);
    if (f != cache.end()) return f->second;
    int per = 0, dev = 0, cus = 0;
    const bool queried =
        hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        (kind == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, lik_persist_kernel<2>,
                                                                  kTileBS, lds)
                   : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, lik_persist_kernel<1>,
                                                                  kTileBS, lds)) == hipSuccess;
    if (!queried) return 0;  // not cached: the next call asks again
    const unsigned cap = (unsigned)std::max(0, per) * (unsigned)std::max(0, cus);
    cache[key] = cap;
    return cap;
}

bool launch_persist(hipStream_t s, const PersistLaunch &p, unsigned blocks)
{
    const unsigned lds = p.t.tab_lds_facet * kRecBytes;
    void *args[] = {const_cast<PersistLaunch *>(&p)};
    const void *fn = p.t.grid == 2 ? (const void *)lik_persist_kernel<2>
                                   : (const void *)lik_persist_kernel<1>;
    return hipLaunchCooperativeKernel(fn, dim3(blocks), dim3(kTileBS), args, lds, s) ==
           hipSuccess;
}

// Fused Newton passes on facets wider than kRecFacet (up to kWideFacet columns): a 24-byte
// record {X, ctr} per column in LDS, and the row-table entries of the rows the work-group's
// chunk spans in a small cache (entry `span` holds row 0, which the zero pad cell reads;
// a span beyond the cache evaluates the row entries per cell from the run tables).  Cell
// ids from cid; the arithmetic and its order are tile_sums64_tab's.
constexpr unsigned kWideRows = 256;
struct ColEntry {
    double xr, xi, c;
};
// The cell centres as the column records hold them (ColEntry::c).
struct ColCtr {
    const ColEntry *col;
    __device__ double operator[](unsigned k) const { return col[k].c; }
};
template <bool CACHED, class Stage>
__device__ inline bool tile_sums64_col(const FacetDev &F, const LikItem &it, double ro,
                                       const Stage &stage, const ColEntry *col,
                                       const double2 *sY, const TabRot<128> &R,
                                       unsigned row_lo, unsigned span, unsigned beg,
                                       unsigned end, double (&s)[7])
{
    const double e1 = it.e1, e2 = it.e2;
    const double detA = 1. - e1 * e1 - e2 * e2;
    const double scale = arcs2rad_scale(ro);
    const double sf = (scale * scale) / (detA * detA);
    const double sw = sf * (4 * kPi * kPi);
    const double a1 = 1. + e1, a2 = 1. - e1;
#pragma unroll
    for (int j = 0; j < 7; j++) s[j] = 0.;
    const uint32_t *cid = F.cid;
    const double2 *dc = F.dc;
    const unsigned pad = F.n;
    auto fetch = [&](RecCells &b, unsigned base) {
#pragma unroll
        for (int q = 0; q < kTabU; q++) {
            const unsigned i = base + q * kTileBS;
            const unsigned k = i < end ? i : pad;
            b.o[q] = gload(cid, k);
            const double2 d = gload(dc, k);
            b.dr[q] = d.x;
            b.di[q] = d.y;
        }
    };
    auto eval = [&](const RecCells &b) {
        double uu[kTabU], vv[kTabU];
        double2 x[kTabU], y[kTabU];
#pragma unroll
        for (int q = 0; q < kTabU; q++) {
            const unsigned ci = b.o[q] & 0xffffu, cj = b.o[q] >> 16;
            const ColEntry &cc = col[ci];
            uu[q] = cc.c;
            vv[q] = col[cj].c;
            x[q] = make_double2(cc.xr, cc.xi);
            // rows below row_lo (only row 0, the pad cell's) wrap past span: entry span
            y[q] = CACHED ? sY[min(cj - row_lo, span)] : tab_y(R, cj);
        }
#pragma unroll
        for (int q = 0; q < kTabU; q++) {
            const double k1 = fma(e2, vv[q], a1 * uu[q]);
            const double k2 = fma(a2, vv[q], e2 * uu[q]);
            const double rr = rsqrt_ge1(fma(sw, fma(k1, k1, k2 * k2), 1.));
            const double M = rr * rr * rr;
            const double hr = b.dr[q] * M;
            const double hi = -b.di[q] * M;
            const double cs = fma(x[q].x, y[q].x, -(x[q].y * y[q].y));
            const double sn = fma(x[q].y, y[q].x, x[q].x * y[q].y);
            const double re = fma(hr, cs, -hi * sn);
            const double im = fma(hr, sn, hi * cs);
            s[0] += re;
            s[1] = fma(-im, uu[q], s[1]);
            s[2] = fma(-im, vv[q], s[2]);
            const double rU = re * uu[q];
            s[3] = fma(-rU, uu[q], s[3]);
            s[4] = fma(-re * vv[q], vv[q], s[4]);
            s[5] = fma(-rU, vv[q], s[5]);
        }
    };
    constexpr unsigned S = kTabU * kTileBS;
    RecCells A, B;
    fetch(A, beg + threadIdx.x);
    if (!stage()) return false;
#pragma unroll
    for (int q = 0; q < kTabU; q++) asm volatile("" : "+v"(A.o[q]), "+v"(A.dr[q]), "+v"(A.di[q]));
    for (unsigned base = beg + threadIdx.x; base < end; base += 2 * S) {
        fetch(B, base + S);
        __builtin_amdgcn_sched_barrier(0);
        eval(A);
        if (base + S >= end) break;
        fetch(A, base + 2 * S);
        __builtin_amdgcn_sched_barrier(0);
        eval(B);
    }
    s[1] *= kTwoPi;
    s[2] *= kTwoPi;
    constexpr double kTwoPi2 = kTwoPi * kTwoPi;
    s[3] *= kTwoPi2;
    s[4] *= kTwoPi2;
    s[5] *= kTwoPi2;
    return true;
}

template <int KIND>
__global__ __launch_bounds__(kTileBS, kTileGridWaves) void lik_fused_wide_kernel(TileLaunch t)
{
    __shared__ double red[(kTileBS / 64) * 8];
    __shared__ int s_go;
    __shared__ double s_off[2];
    __shared__ TabRot<128> R;  // gf <= kWideFacet < 128 runs of kTabRun
    const unsigned per = (t.nwg + kXcds - 1) / kXcds;
    const unsigned wg = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (wg >= t.nwg) return;
    const LikLaunch &a = t.lk;
    const LikItem *items = KIND == 2 ? t.inl : a.items;
    int item;
    unsigned first, nch;
    tile_locate(t, items, wg, &item, &first, &nch);
    const unsigned local = wg - first;
    const unsigned chunk = local / (unsigned)t.nr_g;
    const int r = (int)(local - chunk * (unsigned)t.nr_g) + t.r_lo;
    const FusedPre pre = fused_pre(t, first, nch, item, r);
    const LikItem it = items[item];
    const FacetDev &F = a.facets[it.slot];
    const unsigned beg = chunk * it.chunk_cells;
    const unsigned end = min(F.n, beg + it.chunk_cells);
    const unsigned gf = F.grid_facet;
    // t.tab_lds_facet (rounded up to even) column records, then kWideRows row entries
    extern __shared__ double2 tab_lds[];
    ColEntry *col = reinterpret_cast<ColEntry *>(tab_lds);
    double2 *sY = tab_lds + (size_t)((t.tab_lds_facet + 1) & ~1u) * 3 / 2;
    const uint32_t *cid = F.cid;
    const double *ctr = F.ctr;
    const unsigned row_lo = end > beg ? gload(cid, beg) >> 16 : 0u;
    const unsigned row_hi = end > beg ? gload(cid, end - 1) >> 16 : 0u;
    const unsigned span = row_hi - row_lo + 1;
    const bool cached = span < kWideRows;  // entry span holds row 0
    auto make = [&]() -> bool {
        if (fused_idle(t, chunk, item, r, pre)) return false;
        fused_step(t, first, nch, chunk, item, r, pre, &s_go, s_off);
        // the records' centres do not depend on the step: stored by waves 1.. while wave 0
        // takes it, and the tables read their runs' centres from them
        if (threadIdx.x >= 64)
            for (unsigned k = threadIdx.x - 64; k < gf; k += kTileBS - 64)
                col[k].c = gload(ctr, k);
        __syncthreads();
        if (!s_go) return false;
        const unsigned yb0 = row_lo / kTabRun, yb1 = row_hi / kTabRun;
        tab_rot_stage(R, ColCtr{col}, gf, s_off[0], s_off[1], yb0, yb1, yb0 > 0);
        __syncthreads();
        for (unsigned k = threadIdx.x; k < gf; k += kTileBS) {
            const double2 x = tab_x(R, k);
            col[k].xr = x.x;
            col[k].xi = x.y;
        }
        if (cached)
            for (unsigned q = threadIdx.x; q <= span; q += kTileBS)
                sY[q] = tab_y(R, q < span ? row_lo + q : 0u);
        __syncthreads();
        return true;
    };
    double s[7];
    const bool ran =
        cached ? tile_sums64_col<true>(F, it, a.rg.ro[r], make, col, sY, R, row_lo, span, beg,
                                       end, s)
               : tile_sums64_col<false>(F, it, a.rg.ro[r], make, col, sY, R, row_lo, span, beg,
                                        end, s);
    if (ran) tile_reduce(s, red, t.partials + (size_t)wg * 8);
}

void launch_tile_fused(hipStream_t s, const TileLaunch &t)
{
    const unsigned g = tile_grid(t.nwg, 0);
    if (t.tab_lds_facet > kRecFacet) {
        const unsigned lds =
            ((t.tab_lds_facet + 1) & ~1u) * (unsigned)sizeof(ColEntry) + kWideRows * 16;
        if (t.grid == 2)
            lik_fused_wide_kernel<2><<<g, kTileBS, lds, s>>>(t);
        else
            lik_fused_wide_kernel<1><<<g, kTileBS, lds, s>>>(t);
        return;
    }
    const unsigned lds = t.tab_lds_facet * kRecBytes;
    if (t.grid == 2)
        lik_fused_kernel<2><<<g, kTileBS, lds, s>>>(t);
    else
        lik_fused_kernel<1><<<g, kTileBS, lds, s>>>(t);
}

// Pass 0 on extracted facets with TPW scalelength tasks per work-group (tasks r_lo + TPW g ..
// of one item and chunk; the last group holds what is left): they share each cell's loads,
// centres and shape terms (tile_sums64_p0_db<NT>), and each task's chunk sums go where its
// own work-group of lik_tile_kernel<0, KIND> puts them, with the same values bit for bit.
// Logical work-group wg2 = chunk * groups + g (chunk counted over the launch's items), in the
// XCD-aware order of lik_tile_kernel.
template <int KIND, int NTT>
__device__ inline void p0_group_chunk(const TileLaunch &t, const LikItem *items, int item,
                                      unsigned cg, unsigned chunk, int ra, double *red)
{
    const LikLaunch &a = t.lk;
    const LikItem it = items[item];
    const FacetDev &F = a.facets[it.slot];
    const unsigned beg = chunk * it.chunk_cells;
    const unsigned end = min(F.n, beg + it.chunk_cells);
    extern __shared__ double2 tab_lds[];
    double *sC = reinterpret_cast<double *>(tab_lds);  // tab_lds_facet * 8 bytes
    auto stage = [&]() {
        for (unsigned k = threadIdx.x; k < F.grid_facet; k += kTileBS) sC[k] = gload(F.ctr, k);
        __syncthreads();
    };
    constexpr int NT = NTT;
    double ro[NT];
#pragma unroll
    for (int q = 0; q < NT; q++) ro[q] = a.rg.ro[ra + q];
    double s[NT][7];
    tile_sums64_p0_db<NT>(F, it, ro, sC, stage, beg, end, s);
    const size_t w0 = (size_t)cg * (unsigned)t.nr_g + (unsigned)(ra - t.r_lo);
#pragma unroll
    for (int q = 0; q < NT; q++) tile_reduce(s[q], red, t.partials + (w0 + q) * 8);
}

template <int KIND, int TPW>
__global__ __launch_bounds__(kTileBS, kTileGridWaves) void lik_p0_group_kernel(TileLaunch t)
{
    __shared__ double red[(kTileBS / 64) * 8];
    if (KIND == 2 && blockIdx.x == 0 && threadIdx.x < t.n_inl)
        t.items_w[threadIdx.x] = t.inl[threadIdx.x];
    const LikItem *items = KIND == 2 ? t.inl : t.lk.items;
    const unsigned nr = (unsigned)t.nr_g, groups = (nr + TPW - 1) / TPW;
    const unsigned nwg2 = t.nwg / nr * groups;
    const unsigned per = (nwg2 + kXcds - 1) / kXcds;
    const unsigned nbx = gridDim.x / kXcds;
    for (unsigned j = blockIdx.x / kXcds; j < per; j += nbx) {
        const unsigned wg2 = (blockIdx.x % kXcds) * per + j;
        if (wg2 >= nwg2) break;
        const unsigned cg = wg2 / groups, g = wg2 - cg * groups;
        const int item = t.item_chunks ? (int)(cg / t.item_chunks)
                                       : tile_item(items, t.lk.nitems, cg * nr, (int)nr);
        const unsigned c0 = t.item_chunks ? (unsigned)item * t.item_chunks
                                          : items[item].chunk_first;
        const int ra = t.r_lo + TPW * (int)g;
        const unsigned left = nr - TPW * g;
        if (left >= (unsigned)TPW)
            p0_group_chunk<KIND, TPW>(t, items, item, cg, cg - c0, ra, red);
        else if (TPW == 3 && left == 2)
            p0_group_chunk<KIND, 2>(t, items, item, cg, cg - c0, ra, red);
        else
            p0_group_chunk<KIND, 1>(t, items, item, cg, cg - c0, ra, red);
    }
}

void launch_tile_sums(hipStream_t s, const TileLaunch &t, int pass)
{
    const unsigned g = tile_grid(t.nwg, tuning().tile_blocks);
    if (pass == 0) {
        const unsigned lds = t.tab_lds_facet * 8;
        // the grid kernels' pass 0 with RL2_TUNE_P0_TASKS tasks per work-group (default 3)
        const unsigned tpw = (unsigned)tuning().p0_tasks;
        const unsigned g2 = tile_grid(
            t.nwg / (unsigned)t.nr_g * (((unsigned)t.nr_g + tpw - 1) / tpw), tuning().tile_blocks);
        if (t.grid && tpw == 3) {
            if (t.grid == 2)
                lik_p0_group_kernel<2, 3><<<g2, kTileBS, lds, s>>>(t);
            else
                lik_p0_group_kernel<1, 3><<<g2, kTileBS, lds, s>>>(t);
        } else if (t.grid && tpw == 2) {
            if (t.grid == 2)
                lik_p0_group_kernel<2, 2><<<g2, kTileBS, lds, s>>>(t);
            else
                lik_p0_group_kernel<1, 2><<<g2, kTileBS, lds, s>>>(t);
        } else if (t.grid == 2)
            lik_tile_kernel<0, 2><<<g, kTileBS, lds, s>>>(t);
        else if (t.grid == 1)
            lik_tile_kernel<0, 1><<<g, kTileBS, lds, s>>>(t);
        else
            lik_tile_kernel<0, 0><<<g, kTileBS, lds, s>>>(t);
    } else {
        const unsigned lds = t.tab ? t.tab_lds_facet * (t.tab_y_lds ? 40 : 24) : 0;
        if (t.grid == 2)
            lik_tile_kernel<1, 2><<<g, kTileBS, lds, s>>>(t);
        else if (t.grid == 1)
            lik_tile_kernel<1, 1><<<g, kTileBS, lds, s>>>(t);
        else
            lik_tile_kernel<1, 0><<<g, kTileBS, lds, s>>>(t);
    }
}

void launch_tile_step(hipStream_t s, const TileLaunch &t, int pass)
{
    const unsigned ntask = (unsigned)t.lk.nitems * t.nr_g;
    // the step is wave 0's; the other waves only write the next pass's tables, so a step
    // without tables (the one after an evaluation's last fused pass) runs one wave
    const unsigned bs = t.tab ? kStepBS : 64u;
    if (pass == 0)
        lik_step_kernel<0><<<ntask, bs, 0, s>>>(t);
    else
        lik_step_kernel<1><<<ntask, bs, 0, s>>>(t);
}

void launch_tile_pass(hipStream_t s, const TileLaunch &t, int pass)
{
    launch_tile_sums(s, t, pass);
    launch_tile_step(s, t, pass);
}

void launch_rmarg(hipStream_t s, const LikLaunch &a)
{
    if (a.nitems <= 0) return;
    rmarg_kernel<<<a.nitems + (a.status ? 1 : 0), 128, 0, s>>>(a);
}

__global__ void marginalise_r_kernel(int num, const double *x, const double *y, double *out,
                                     double *ws, int *iws)
{
    double xx[kMaxR], yy[kMaxR];
    for (int i = 0; i < num; i++) {
        xx[i] = x[i];
        yy[i] = y[i];
    }
    QagWs w{ws, ws + kQagLimit, ws + 2 * kQagLimit, ws + 3 * kQagLimit, iws, iws + kQagLimit};
    out[0] = marginalise_posterior(num, xx, yy, w);
    for (int i = 0; i < num; i++) out[1 + i] = yy[i];
}

void launch_marginalise_r(hipStream_t s, int num, const double *x, const double *y,
                          double *out, double *qag_ws, int *qag_iws)
{
    marginalise_r_kernel<<<1, 1, 0, s>>>(num, x, y, out, qag_ws, qag_iws);
}

// marg_position (likelihood.c:376-421) on n given arguments, the same bits either way: one per
// wave, the device function finish_lr applies to B = ho^2 / 2, or one per lane.
__global__ __launch_bounds__(64) void marg_position_kernel(int n, const double *x, double *out)
{
    const int i = blockIdx.x;
    const double y = marg_position_wave(x[i]);
    if (threadIdx.x == 0) out[i] = y;
}
__global__ __launch_bounds__(256) void marg_position_lanes_kernel(int n, const double *x,
                                                                  double *out)
{
    const int i = (int)(blockIdx.x * 256u + threadIdx.x);
    if (i < n) out[i] = marg_position(x[i]);
}

// A wave ends an argument soonest, lanes take more of them at a time, and a launch holds fewer
// than 2^26 waves: whole calls by waves / lanes take 33 / 60 us for 100 arguments, 110 / 114 for
// 8,192, 147 / 144 for 12,288, 86 / 70 for 16,384 (another kind of copy) and 3,000 / 1,020 for a
// million.
void launch_marg_position(hipStream_t s, int n, const double *x, double *out)
{
    constexpr int kMargLanes = 10240;
    if (n <= 0) return;
    if (n < kMargLanes)
        marg_position_kernel<<<n, 64, 0, s>>>(n, x, out);
    else
        marg_position_lanes_kernel<<<((unsigned)n + 255u) / 256u, 256, 0, s>>>(n, x, out);
}

// ------------------------------------------------------------------ subtraction (K2)
// data_processing.c:109-135: visSkyMod -= round model, visData -= fitted model, i.e.
// R = (R - fit) + round with one phase rotor per visibility.
template <int PREC>
__global__ __launch_bounds__(256) void subtract_kernel(unsigned nch, unsigned long nrow,
                                                       const double *__restrict__ u,
                                                       const double *__restrict__ v,
                                                       const double *__restrict__ w,
                                                       const double *__restrict__ wn,
                                                       const double *__restrict__ inv_lambda,
                                                       const double *__restrict__ spec,
                                                       GalaxyGeom fit, GalaxyGeom rnd, void *res)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nrow) return;
    const double ui = u[i], vi = v[i], wi = w[i];
    const double p = ui * fit.l0 + vi * fit.m0 + wi * fit.n0;
    for (unsigned c = 0; c < nch; c++) {
        const double k = wn[c], k2 = k * k, spectra = spec[c];
        const size_t idx = (size_t)c * nrow + i;
        const double2 r = subtract_vis(fit, rnd, p, ui, vi, k2, spectra, inv_lambda[c],
                                       load_res(res, PREC, idx));
        store_res(res, PREC, idx, r);
    }
}

void launch_subtract(hipStream_t s, int prec, unsigned nch, unsigned long nrow, const double *u,
                     const double *v, const double *w, const double *wn,
                     const double *inv_lambda, const double *spec,
                     const GalaxyGeom &fit, const GalaxyGeom &round, void *res)
{
    dim3 grid((unsigned)((nrow + 255) / 256));
    if (prec == 0)
        subtract_kernel<0><<<grid, 256, 0, s>>>(nch, nrow, u, v, w, wn, inv_lambda, spec, fit,
                                                 round, res);
    else
        subtract_kernel<1><<<grid, 256, 0, s>>>(nch, nrow, u, v, w, wn, inv_lambda, spec, fit,
                                                 round, res);
}

// ------------------------------------------------------------------ drop-in helpers
// galaxy_visibilities.c:59-91 in two steps: model + per-block partial sums of M^2/sigma^2,
// then normalisation by sqrt of the fixed-order total.
__global__ __launch_bounds__(256) void model_zero_kernel(double e1, double e2, double sf, unsigned n,
                                                         const double *uu, const double *vv,
                                                         const double *s2, double *mod,
                                                         double *partials)
{
    __shared__ double red[4];
    unsigned i = blockIdx.x * 256 + threadIdx.x;
    double t = 0.;
    if (i < n) {
        double k1 = (1. + e1) * uu[i] + e2 * vv[i];
        double k2 = e2 * uu[i] + (1. - e1) * vv[i];
        double M = sersic_shape(k1, k2, sf, 4 * kPi * kPi);
        mod[i] = M;
        t = M * M / s2[i];
    }
    double v[1] = {t};
    block_allreduce<256, 1>(v, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = v[0];
}
__global__ __launch_bounds__(256) void model_norm_kernel(unsigned n, unsigned nb,
                                                         const double *partials, double *mod)
{
    __shared__ double tot;
    if (threadIdx.x == 0) {
        double s = 0.;
        for (unsigned b = 0; b < nb; b++) s += partials[b];
        tot = sqrt(s);
    }
    __syncthreads();
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) mod[i] /= tot;
}
void launch_model_at_zero(hipStream_t s, double e1, double e2, double scale, unsigned n,
                          const double *uu, const double *vv, const double *s2, double *mod,
                          double *partials)
{
    double detA = 1. - e1 * e1 - e2 * e2;
    double sc = arcs2rad_scale(scale);
    double sf = (sc * sc) / (detA * detA);
    unsigned nb = (n + 255) / 256;
    if (nb == 0) return;
    model_zero_kernel<<<nb, 256, 0, s>>>(e1, e2, sf, n, uu, vv, s2, mod, partials);
    model_norm_kernel<<<min(nb, 1024u), 256, 0, s>>>(n, nb, partials, mod);
}

__global__ void galaxy_vis_kernel(double spectra, double wn, GalaxyGeom g, unsigned long n,
                                  const double *u, const double *v, const double *w, double *vis)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double ui = u[i], vi = v[i], wi = w[i];
    double phase = ui * g.l0 + vi * g.m0 + wi * g.n0;
    phase = wn * phase;
    double shape = model_shape(g, ui, vi, wn * wn, spectra);
    double sn, cs;
    sincos(phase, &sn, &cs);
    vis[2 * i] = shape * cs;
    vis[2 * i + 1] = shape * sn;
}
void launch_galaxy_vis(hipStream_t s, double spectra, double wavenumber, const GalaxyGeom &g,
                       unsigned long n, const double *u, const double *v, const double *w,
                       double *vis)
{
    if (!n) return;
    galaxy_vis_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(spectra, wavenumber, g, n, u, v,
                                                                  w, vis);
}

__global__ void phase_shift_kernel(double wn, double l, double m, double nn, unsigned long n,
                                   const double *u, const double *v, const double *w, double *vis)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double phase = u[i] * l + v[i] * m + w[i] * nn;
    phase *= -wn;
    double sp, cp;
    sincos(phase, &sp, &cp);
    double re = vis[2 * i], im = vis[2 * i + 1];
    vis[2 * i] = re * cp - im * sp;
    vis[2 * i + 1] = re * sp + im * cp;
}
void launch_phase_shift(hipStream_t s, double wavenumber, double l, double m, unsigned long n,
                        const double *u, const double *v, const double *w, double *vis)
{
    if (!n) return;
    double nn = sqrt(1. - l * l - m * m) - 1.;
    phase_shift_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(wavenumber, l, m, nn, n, u, v,
                                                                   w, vis);
}

// ------------------------------------------------------------------ observation set-up
__global__ void gather_rows_kernel(unsigned long nrow, const uint32_t *perm, const double *src,
                                   double *dst)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i < nrow) dst[i] = src[perm[i]];
}
void launch_gather_rows(hipStream_t s, unsigned long nrow, const uint32_t *perm,
                        const double *src, double *dst)
{
    gather_rows_kernel<<<(unsigned)((nrow + 255) / 256), 256, 0, s>>>(nrow, perm, src, dst);
}

__global__ void pack_sigma_kernel(unsigned nch, unsigned long nrow, const uint32_t *perm,
                                  const float *sigma2, const unsigned char *flag, float *s2f)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nrow) return;
    unsigned long src = perm[i];
    for (unsigned c = 0; c < nch; c++) {
        float sg = sigma2[(size_t)c * nrow + src];
        bool fl = flag && flag[(size_t)c * nrow + src];
        if (isnan(sg) && !signbit(sg)) sg = 0.f;  // adds nothing, as its conversion did
        s2f[(size_t)c * nrow + i] = fl ? -fabsf(sg) - 0.0f : sg;
    }
}
void launch_pack_sigma(hipStream_t s, unsigned nch, unsigned long nrow, const uint32_t *perm,
                       const float *sigma2, const unsigned char *flag, float *s2f)
{
    pack_sigma_kernel<<<(unsigned)((nrow + 255) / 256), 256, 0, s>>>(nch, nrow, perm, sigma2, flag,
                                                                     s2f);
}

template <int PREC>
__global__ void residual_in_kernel(unsigned nch, unsigned long nrow, const uint32_t *perm,
                                   const double *D, const double *S, void *res)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nrow) return;
    unsigned long src = perm[i];
    for (unsigned c = 0; c < nch; c++) {
        size_t k = (size_t)c * nrow + src;
        double re = D[2 * k], im = D[2 * k + 1];
        if (S) {
            re = re - S[2 * k];
            im = im - S[2 * k + 1];
        }
        store_res(res, PREC, (size_t)c * nrow + i, make_double2(re, im));
    }
}
void launch_residual_in(hipStream_t s, int prec, unsigned nch, unsigned long nrow,
                        const uint32_t *perm, const double *D, const double *S, void *res)
{
    dim3 grid((unsigned)((nrow + 255) / 256));
    if (prec == 0)
        residual_in_kernel<0><<<grid, 256, 0, s>>>(nch, nrow, perm, D, S, res);
    else
        residual_in_kernel<1><<<grid, 256, 0, s>>>(nch, nrow, perm, D, S, res);
}

template <int PREC>
__global__ void residual_out_kernel(unsigned nch, unsigned long nrow, const uint32_t *perm,
                                    const void *res, double *out)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nrow) return;
    unsigned long dst = perm[i];
    for (unsigned c = 0; c < nch; c++) {
        double2 r = load_res(res, PREC, (size_t)c * nrow + i);
        size_t k = (size_t)c * nrow + dst;
        out[2 * k] = r.x;
        out[2 * k + 1] = r.y;
    }
}
void launch_residual_out(hipStream_t s, int prec, unsigned nch, unsigned long nrow,
                         const uint32_t *perm, const void *res, double *out)
{
    dim3 grid((unsigned)((nrow + 255) / 256));
    if (prec == 0)
        residual_out_kernel<0><<<grid, 256, 0, s>>>(nch, nrow, perm, res, out);
    else
        residual_out_kernel<1><<<grid, 256, 0, s>>>(nch, nrow, perm, res, out);
}

// Morton (Z-order) key of (u, v) quantised to 16 bits per axis over [-umax, umax].
__device__ inline uint32_t spread16(uint32_t x)
{
    x &= 0xffffu;
    x = (x | (x << 8)) & 0x00ff00ffu;
    x = (x | (x << 4)) & 0x0f0f0f0fu;
    x = (x | (x << 2)) & 0x33333333u;
    x = (x | (x << 1)) & 0x55555555u;
    return x;
}
__global__ void morton_kernel(unsigned long nrow, const double *u, const double *v, double umax,
                              uint32_t *keys, uint32_t *idx)
{
    unsigned long i = blockIdx.x * (unsigned long)blockDim.x + threadIdx.x;
    if (i >= nrow) return;
    double s = 65535.0 / (2.0 * umax);
    double qu = fmin(fmax((u[i] + umax) * s, 0.0), 65535.0);
    double qv = fmin(fmax((v[i] + umax) * s, 0.0), 65535.0);
    keys[i] = spread16((uint32_t)qu) | (spread16((uint32_t)qv) << 1);
    idx[i] = (uint32_t)i;
}
void launch_morton_keys(hipStream_t s, unsigned long nrow, const double *u, const double *v,
                        double umax, uint32_t *keys, uint32_t *idx)
{
    morton_kernel<<<(unsigned)((nrow + 255) / 256), 256, 0, s>>>(nrow, u, v, umax, keys, idx);
}

size_t sort_rows_tmp_bytes(unsigned long nrow)
{
    size_t bytes = 0;
    hipcub::DoubleBuffer<uint32_t> k(nullptr, nullptr), v(nullptr, nullptr);
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k, v, (int)nrow) != hipSuccess)
        return 0;  // the sort itself then reports the failure
    return bytes;
}

bool sort_rows(hipStream_t s, unsigned long nrow, uint32_t *keys, uint32_t *idx,
               uint32_t *keys_alt, uint32_t *idx_alt, void *tmp, size_t tmp_bytes,
               uint32_t **sorted_idx)
{
    hipcub::DoubleBuffer<uint32_t> k(keys, keys_alt), v(idx, idx_alt);
    const bool ok = hip_ok(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, k, v, (int)nrow,
                                                              0, 32, s),
                           "row sort");
    *sorted_idx = v.Current();
    return ok;
}

}  // namespace rl2
