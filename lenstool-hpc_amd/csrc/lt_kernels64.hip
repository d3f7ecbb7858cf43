// lt_kernels64.hip -- FP64 lens-map kernels for gfx950: gradient, Hessian (+ fused map epilogue),
// potential. One thread owns PX pixels of one row (columns lane, lane+64, ...); a 64x4 workgroup
// covers 64*PX columns of 4 rows. Halo records are walked in wavefront-uniform order, run by run.
//
// Small maps leave most of the chip idle that way: 200 x 200 pixels are 313 waves of two pixels a lane for
// 1024 SIMDs, each walking every halo one record load after another. The split form (SUM_WAVES) gives a
// row segment of 64 PX pixels to kSplit waves, wave s taking halos s, s + kSplit, .. of the model (so that every
// wave has its share of each type), and adds their sums through LDS in the order of the waves. A batch of small
// maps fills the chip with a wave per segment: SUM_PARTS forms the same parts and sums one after another.
//
// Formulas (restated from the mathematics; reference equivalents cited):
//   SIS gradient  src/gradient.cpp:260-299      PIEMD gradient  src/gradient.hpp:64-76,
//   dPIE gradient src/gradient.cpp:744-809      PIEMD Hessian   src/gradient2.cpp:54-82, 92-205
//   potential     src/potential_GPU.cu:47-116   epilogues       src/grid_map_*_GPU.cu
#include <hip/hip_runtime.h>

#include "lenstool_hip/lt_status.h"
#include "lt_device.h"
#include "lt_kernels.h"
#include "lt_math.h"
#include "lt_terms64.h"

namespace lt {

// part `wave` of SPLIT of the Hessian sums at PX pixels of a row, run by run. UNIT: every run's weight is 1 and its terms
// are added to the part's sums as they come, with no sums of the run's own.
template <int PX, int SPLIT, bool UNIT>
__device__ __forceinline__ void hessian_sums(const HaloRec* __restrict__ halos, const Run* __restrict__ runs, int nruns,
                                             int wave, const double* px, double py, double* tT, double* tD, double* tB)
{
#pragma unroll
    for (int k = 0; k < PX; ++k) tT[k] = tD[k] = tB[k] = 0.;
    for (int r = 0; r < nruns; ++r) {
        const Run run = runs[r];
        if (SPLIT > 1 && first_halo<SPLIT>(run.start, wave) >= run.start + run.count) continue;
        double rT[PX], rD[PX], rB[PX];
        double *const sT = UNIT ? tT : rT, *const sD = UNIT ? tD : rD, *const sB = UNIT ? tB : rB;
#pragma unroll
        for (int k = 0; k < PX; ++k) rT[k] = rD[k] = rB[k] = 0.;
        const int end = run.start + run.count;
        switch (run.type) {
        case TYPE_DPIE:
            for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                const HaloRec& h = halos[i];
#pragma unroll
                for (int k = 0; k < PX; ++k) hess_piemd<true>(h, px[k], py, sT[k], sD[k], sB[k]);
            }
            break;
        case TYPE_PIEMD:
            for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                const HaloRec& h = halos[i];
#pragma unroll
                for (int k = 0; k < PX; ++k) hess_piemd<false>(h, px[k], py, sT[k], sD[k], sB[k]);
            }
            break;
        case TYPE_SIS:
            if (run.circ) {
                // four halos per step: their records' scalar loads issue together, one wait per step
#pragma unroll 4
                for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                    const HaloRec& h = halos[i];
#pragma unroll
                    for (int k = 0; k < PX; ++k) hess_sis_circ(h, px[k], py, sT[k], sD[k], sB[k]);
                }
            } else {
                for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                    const HaloRec& h = halos[i];
#pragma unroll
                    for (int k = 0; k < PX; ++k) hess_sis(h, px[k], py, sT[k], sD[k], sB[k]);
                }
            }
            break;
        default:  // TYPE_SHEAR: constant lab-frame Hessian
            for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                const HaloRec& h = halos[i];
#pragma unroll
                for (int k = 0; k < PX; ++k) {
                    sT[k] += h.h14a + h.h14c;
                    sD[k] += h.h14a - h.h14c;
                    sB[k] += h.h14b;
                }
            }
            break;
        }
        if (UNIT) continue;
        const double w = run.weight;
#pragma unroll
        for (int k = 0; k < PX; ++k) {
            tT[k] = __builtin_fma(w, sT[k], tT[k]);
            tD[k] = __builtin_fma(w, sD[k], tD[k]);
            tB[k] = __builtin_fma(w, sB[k], tB[k]);
        }
    }
}

template <int PX, int KIND, int FORM, bool UNIT>
__global__ __launch_bounds__(WAVE* rows_of(FORM), FORM == SUM_PARTS && PX == 2 ? 5 : 1) void k_hessian64(const HaloRec* __restrict__ halos,
                                                                   const Run* __restrict__ runs, int nruns, GridDesc g,
                                                                   OutDesc o)
{
    const int wave = FORM == SUM_WAVES ? __builtin_amdgcn_readfirstlane(threadIdx.y) : 0;
    const int row = FORM == SUM_WAVES ? blockIdx.y : blockIdx.y * ROWS + threadIdx.y;
    if (row >= g.ny) return;
    halos = select_sample(g, halos, o);
    const int col0 = blockIdx.x * (WAVE * PX) + threadIdx.x;
    const double py = pixel_coord(g.ymin, row + g.jstart, g.dy);
    double px[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) px[k] = pixel_coord(g.xmin, col0 + k * WAVE + g.istart, g.dx);
    double tT[PX], tD[PX], tB[PX];
    if constexpr (FORM == SUM_PARTS) {
#pragma unroll
        for (int k = 0; k < PX; ++k) tT[k] = tD[k] = tB[k] = 0.;
#pragma unroll 1
        for (int m = g.parts; m; m &= m - 1) {
            double sT[PX], sD[PX], sB[PX];
            hessian_sums<PX, kSplit, UNIT>(halos, runs, nruns, __builtin_ctz(m), px, py, sT, sD, sB);
            add_part<PX>(tT, sT);
            add_part<PX>(tD, sD);
            add_part<PX>(tB, sB);
        }
    } else {
        hessian_sums<PX, parts_of(FORM), UNIT>(halos, runs, nruns, wave, px, py, tT, tD, tB);
    }
    if constexpr (FORM == SUM_WAVES) {
        if constexpr (KIND == LT_MAP_MASS) {
            if (!split_sum<PX, kSplit>(wave, tT)) return;
        } else {
            if (!split_sum<PX, kSplit>(wave, tT, tD, tB)) return;
        }
        const int col = col0 + wave * WAVE;
        if (col < g.nx) hess_epilogue<KIND>(o, (int64_t)row * g.pitch + col, tT[0], tD[0], tB[0]);
        return;
    }
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        const int col = col0 + k * WAVE;
        if (col < g.nx) hess_epilogue<KIND>(o, (int64_t)row * g.pitch + col, tT[k], tD[k], tB[k]);
    }
}

// the same of the gradient sums
template <int PX, int SPLIT>
__device__ __forceinline__ void gradient_sums(const HaloRec* __restrict__ halos, const Run* __restrict__ runs, int nruns,
                                              int wave, const double* px, double py, double* tx, double* ty)
{
#pragma unroll
    for (int k = 0; k < PX; ++k) tx[k] = ty[k] = 0.;
    for (int r = 0; r < nruns; ++r) {
        const Run run = runs[r];
        if (SPLIT > 1 && first_halo<SPLIT>(run.start, wave) >= run.start + run.count) continue;
        double rx[PX], ry[PX];  // a part's terms are added to its sums as they come
        double *const sx = SPLIT > 1 ? tx : rx, *const sy = SPLIT > 1 ? ty : ry;
#pragma unroll
        for (int k = 0; k < PX; ++k) rx[k] = ry[k] = 0.;
        const int end = run.start + run.count;
        switch (run.type) {
        case TYPE_DPIE:
            for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                const HaloRec& h = halos[i];
#pragma unroll
                for (int k = 0; k < PX; ++k) grad_piemd<true>(h, px[k], py, sx[k], sy[k]);
            }
            break;
        case TYPE_PIEMD:
            for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                const HaloRec& h = halos[i];
#pragma unroll
                for (int k = 0; k < PX; ++k) grad_piemd<false>(h, px[k], py, sx[k], sy[k]);
            }
            break;
        default:  // TYPE_SIS
            if (run.circ) {
                // four halos per step: their records' scalar loads issue together, one wait per step
#pragma unroll 4
                for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                    const HaloRec& h = halos[i];
#pragma unroll
                    for (int k = 0; k < PX; ++k) grad_sis_circ(h, px[k], py, sx[k], sy[k]);
                }
            } else {
                for (int i = first_halo<SPLIT>(run.start, wave); i < end; i += SPLIT) {
                    const HaloRec& h = halos[i];
#pragma unroll
                    for (int k = 0; k < PX; ++k) grad_sis(h, px[k], py, sx[k], sy[k]);
                }
            }
            break;
        }
        if (SPLIT > 1) continue;
#pragma unroll
        for (int k = 0; k < PX; ++k) {
            tx[k] += sx[k];
            ty[k] += sy[k];
        }
    }
}

template <int PX, int FORM>
__global__ __launch_bounds__(WAVE* rows_of(FORM)) void k_gradient64(const HaloRec* __restrict__ halos,
                                                                    const Run* __restrict__ runs, int nruns, GridDesc g,
                                                                    OutDesc o)
{
    const int wave = FORM == SUM_WAVES ? __builtin_amdgcn_readfirstlane(threadIdx.y) : 0;
    const int row = FORM == SUM_WAVES ? blockIdx.y : blockIdx.y * ROWS + threadIdx.y;
    if (row >= g.ny) return;
    halos = select_sample(g, halos, o);
    const int col0 = blockIdx.x * (WAVE * PX) + threadIdx.x;
    const double py = pixel_coord(g.ymin, row + g.jstart, g.dy);
    double px[PX], tx[PX], ty[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) px[k] = pixel_coord(g.xmin, col0 + k * WAVE + g.istart, g.dx);
    if constexpr (FORM == SUM_PARTS) {
#pragma unroll
        for (int k = 0; k < PX; ++k) tx[k] = ty[k] = 0.;
#pragma unroll 1
        for (int m = g.parts; m; m &= m - 1) {
            double sx[PX], sy[PX];
            gradient_sums<PX, kSplit>(halos, runs, nruns, __builtin_ctz(m), px, py, sx, sy);
            add_part<PX>(tx, sx);
            add_part<PX>(ty, sy);
        }
    } else {
        gradient_sums<PX, parts_of(FORM)>(halos, runs, nruns, wave, px, py, tx, ty);
    }
    const double m = o.kind == LT_MAP_DPL ? o.r : 1.0;
    if constexpr (FORM == SUM_WAVES) {
        if (!split_sum<PX, kSplit>(wave, tx, ty)) return;
        const int col = col0 + wave * WAVE;
        if (col < g.nx) {
            const int64_t idx = (int64_t)row * g.pitch + col;
            o.p0[idx] = tx[0] * m;
            o.p1[idx] = ty[0] * m;
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        const int col = col0 + k * WAVE;
        if (col < g.nx) {
            const int64_t idx = (int64_t)row * g.pitch + col;
            o.p0[idx] = tx[k] * m;
            o.p1[idx] = ty[k] * m;
        }
    }
}

// the same of the potential; mn = min(mn, rem^2) over the part's PIEMD and dPIE halos
template <int PX, int SPLIT>
__device__ __forceinline__ void potential_sums(const HaloRec* __restrict__ halos, const Run* __restrict__ runs, int nruns,
                                               int wave, const double* px, double py, double* tot, double* mn)
{
#pragma unroll
    for (int k = 0; k < PX; ++k) tot[k] = 0.;
    for (int r = 0; r < nruns; ++r) {
        const Run run = runs[r];
        if (SPLIT > 1 && first_halo<SPLIT>(run.start, wave) >= run.start + run.count) continue;
        double rs[PX];
        double* const s = SPLIT > 1 ? tot : rs;
#pragma unroll
        for (int k = 0; k < PX; ++k) rs[k] = 0.;
        for (int i = first_halo<SPLIT>(run.start, wave); i < run.start + run.count; i += SPLIT) {
            const HaloRec& h = halos[i];
#pragma unroll
            for (int k = 0; k < PX; ++k) add_pot_halo<false>(h, run.type, px[k] - h.xh, py - h.yh, s[k], mn[k]);
        }
        if (SPLIT > 1) continue;
#pragma unroll
        for (int k = 0; k < PX; ++k) tot[k] += s[k];
    }
}

template <int PX, int FORM>
__global__ __launch_bounds__(WAVE* rows_of(FORM)) void k_potential64(const HaloRec* __restrict__ halos,
                                                                     const Run* __restrict__ runs, int nruns, GridDesc g,
                                                                     OutDesc o)
{
    const int wave = FORM == SUM_WAVES ? __builtin_amdgcn_readfirstlane(threadIdx.y) : 0;
    const int row = FORM == SUM_WAVES ? blockIdx.y : blockIdx.y * ROWS + threadIdx.y;
    if (row >= g.ny) return;
    halos = select_sample(g, halos, o);
    const int col0 = blockIdx.x * (WAVE * PX) + threadIdx.x;
    const double py = pixel_coord(g.ymin, row + g.jstart, g.dy);
    double px[PX], tot[PX], mn[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        px[k] = pixel_coord(g.xmin, col0 + k * WAVE + g.istart, g.dx);
        mn[k] = 1.;
    }
    if constexpr (FORM == SUM_PARTS) {
#pragma unroll
        for (int k = 0; k < PX; ++k) tot[k] = 0.;
#pragma unroll 1
        for (int m = g.parts; m; m &= m - 1) {
            double s[PX];
            potential_sums<PX, kSplit>(halos, runs, nruns, __builtin_ctz(m), px, py, s, mn);
            add_part<PX>(tot, s);
        }
    } else {
        potential_sums<PX, parts_of(FORM)>(halos, runs, nruns, wave, px, py, tot, mn);
    }
    if constexpr (FORM == SUM_WAVES) {
        // a wave that met a PIEMD centre makes the sum NaN
#pragma unroll
        for (int k = 0; k < PX; ++k)
            if (mn[k] == 0.) tot[k] = __builtin_nan("");
        if (!split_sum<PX, kSplit>(wave, tot)) return;
        const int col = col0 + wave * WAVE;
        if (col < g.nx) o.p0[(int64_t)row * g.pitch + col] = tot[0] * o.mult;
        return;
    }
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        const int col = col0 + k * WAVE;
        // a pixel on a PIEMD centre: the reference's potential is 0/0 there
        const double v = mn[k] == 0. ? __builtin_nan("") : tot[k] * o.mult;
        if (col < g.nx) o.p0[(int64_t)row * g.pitch + col] = v;
    }
}

// Gradient at arbitrary points for a batch of lens models (blockIdx.y = sample), e.g. at the
// observed images for the source barycentres: kSplit waves share the halos of 64 points, as in the split maps. Points
// come by the thousand, and one wave per 64 of them walked all halos in a serial chain on a third of the SIMDs: 20000
// points and 503 dPIE halos 290 us, now 78 (the 20M instructions' issue alone is 35; 313 work-groups on 256 CUs leave
// the last ones two deep); 200000 points 25 us less of 720 with their copies, so no second form is kept. Parts of the
// halos over several work-groups and a second kernel for their sum took 54 us here, but the call as a whole 23 more.
__global__ __launch_bounds__(WAVE* kSplit) void k_points_gradient64(const HaloRec* __restrict__ halos,
                                                                   const Run* __restrict__ runs, int nruns,
                                                                   const double* __restrict__ px,
                                                                   const double* __restrict__ py, int npts,
                                                                   int64_t halo_stride, double* __restrict__ gx,
                                                                   double* __restrict__ gy)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int i = blockIdx.x * WAVE + threadIdx.x;
    const int64_t s = blockIdx.y;
    halos += s * halo_stride;
    const int at = min(i, npts - 1);  // every lane takes part in the sums
    const double x = px[at], y = py[at];
    double tx[1] = {0.}, ty[1] = {0.};
    for (int r = 0; r < nruns; ++r) {
        const Run run = runs[r];
        double sx = 0., sy = 0.;
        const int end = run.start + run.count;
        int h = first_halo<kSplit>(run.start, wave);
        switch (run.type) {
        case TYPE_DPIE:
            for (; h < end; h += kSplit) grad_piemd<true>(halos[h], x, y, sx, sy);
            break;
        case TYPE_PIEMD:
            for (; h < end; h += kSplit) grad_piemd<false>(halos[h], x, y, sx, sy);
            break;
        default:
            if (run.circ)
                for (; h < end; h += kSplit) grad_sis_circ(halos[h], x, y, sx, sy);
            else
                for (; h < end; h += kSplit) grad_sis(halos[h], x, y, sx, sy);
            break;
        }
        tx[0] += sx;
        ty[0] += sy;
    }
    if (!split_sum<1, kSplit>(wave, tx, ty) || i >= npts) return;
    const int64_t o = s * npts + i;
    gx[o] = tx[0];
    gy[o] = ty[0];
}

// Epilogue alone, on Hessian planes already in device memory (the reference's map functions
// amplif_k_grid_CPU_GPU & co. work this way, src/grid_map_ampli_GPU.cu:305-547).
template <int KIND>
__global__ __launch_bounds__(256) void k_epilogue(const double* __restrict__ a, const double* __restrict__ b,
                                                  const double* __restrict__ c, int64_t n, OutDesc o)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const double av = a[i], cv = c[i];
        hess_epilogue<KIND>(o, i, av + cv, av - cv, b[i]);
    }
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
template <int PX, int FORM, bool UNIT = false>
static hipError_t launch_hessian64_px(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                                      const OutDesc& o, hipStream_t s)
{
    dim3 blk, grd;
    geometry<PX, FORM>(g, grd, blk);
    switch (o.kind) {
    case LT_MAP_FIELDS: hipLaunchKernelGGL((k_hessian64<PX, LT_MAP_FIELDS, FORM, UNIT>), grd, blk, 0, s, halos, runs, nruns, g, o); break;
    case LT_MAP_AMPLI: hipLaunchKernelGGL((k_hessian64<PX, LT_MAP_AMPLI, FORM, UNIT>), grd, blk, 0, s, halos, runs, nruns, g, o); break;
    case LT_MAP_SHEAR: hipLaunchKernelGGL((k_hessian64<PX, LT_MAP_SHEAR, FORM, UNIT>), grd, blk, 0, s, halos, runs, nruns, g, o); break;
    case LT_MAP_MASS: hipLaunchKernelGGL((k_hessian64<PX, LT_MAP_MASS, FORM, UNIT>), grd, blk, 0, s, halos, runs, nruns, g, o); break;
    default: hipLaunchKernelGGL((k_hessian64<PX, LT_MAP_HESSIAN, FORM, UNIT>), grd, blk, 0, s, halos, runs, nruns, g, o); break;
    }
    return hipGetLastError();
}

hipError_t launch_hessian64(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                            const OutDesc& o, int px, bool unit, hipStream_t s)
{
    switch (px) {
    case kPxSplit:
        return unit ? launch_hessian64_px<1, SUM_WAVES, true>(halos, runs, nruns, g, o, s)
                    : launch_hessian64_px<1, SUM_WAVES>(halos, runs, nruns, g, o, s);
    case kPxParts:
        if (parts_px(g, 1.15) == 1)
            return unit ? launch_hessian64_px<1, SUM_PARTS, true>(halos, runs, nruns, g, o, s)
                        : launch_hessian64_px<1, SUM_PARTS>(halos, runs, nruns, g, o, s);
        return unit ? launch_hessian64_px<2, SUM_PARTS, true>(halos, runs, nruns, g, o, s)
                    : launch_hessian64_px<2, SUM_PARTS>(halos, runs, nruns, g, o, s);
    case 1: return launch_hessian64_px<1, SUM_PLAIN>(halos, runs, nruns, g, o, s);
    case 4: return launch_hessian64_px<4, SUM_PLAIN>(halos, runs, nruns, g, o, s);
    default: return launch_hessian64_px<2, SUM_PLAIN>(halos, runs, nruns, g, o, s);
    }
}

hipError_t launch_epilogue64(const double* a, const double* b, const double* c, int64_t n, const OutDesc& o,
                             hipStream_t s)
{
    int64_t nb = (n + 255) / 256;
    unsigned blocks = (unsigned)(nb > 16384 ? 16384 : (nb ? nb : 1));
    dim3 blk(256), grd(blocks);
    switch (o.kind) {
    case LT_MAP_FIELDS: hipLaunchKernelGGL((k_epilogue<LT_MAP_FIELDS>), grd, blk, 0, s, a, b, c, n, o); break;
    case LT_MAP_AMPLI: hipLaunchKernelGGL((k_epilogue<LT_MAP_AMPLI>), grd, blk, 0, s, a, b, c, n, o); break;
    case LT_MAP_SHEAR: hipLaunchKernelGGL((k_epilogue<LT_MAP_SHEAR>), grd, blk, 0, s, a, b, c, n, o); break;
    case LT_MAP_MASS: hipLaunchKernelGGL((k_epilogue<LT_MAP_MASS>), grd, blk, 0, s, a, b, c, n, o); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_points_gradient64(const HaloRec* halos, const Run* runs, int nruns, const double* px,
                                    const double* py, int npts, int nsamples, int64_t halo_stride, double* gx,
                                    double* gy, hipStream_t s)
{
    hipLaunchKernelGGL(k_points_gradient64, dim3((npts + WAVE - 1) / WAVE, nsamples), dim3(WAVE, kSplit), 0, s, halos,
                       runs, nruns, px, py, npts, halo_stride, gx, gy);
    return hipGetLastError();
}

template <int PX, int FORM>
static void launch_gradient64_px(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g, const OutDesc& o,
                           hipStream_t s)
{
    dim3 blk, grd;
    geometry<PX, FORM>(g, grd, blk);
    hipLaunchKernelGGL((k_gradient64<PX, FORM>), grd, blk, 0, s, halos, runs, nruns, g, o);
}

hipError_t launch_gradient64(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                             const OutDesc& o, int px, hipStream_t s)
{
    switch (px) {
    case kPxSplit: launch_gradient64_px<1, SUM_WAVES>(halos, runs, nruns, g, o, s); break;
    case kPxParts:
        if (parts_px(g, 1.0) == 1) launch_gradient64_px<1, SUM_PARTS>(halos, runs, nruns, g, o, s);
        else launch_gradient64_px<2, SUM_PARTS>(halos, runs, nruns, g, o, s);
        break;
    case 1: launch_gradient64_px<1, SUM_PLAIN>(halos, runs, nruns, g, o, s); break;
    case 4: launch_gradient64_px<4, SUM_PLAIN>(halos, runs, nruns, g, o, s); break;
    default: launch_gradient64_px<2, SUM_PLAIN>(halos, runs, nruns, g, o, s); break;
    }
    return hipGetLastError();
}

template <int PX, int FORM>
static void launch_potential64_px(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g, const OutDesc& o,
                           hipStream_t s)
{
    dim3 blk, grd;
    geometry<PX, FORM>(g, grd, blk);
    hipLaunchKernelGGL((k_potential64<PX, FORM>), grd, blk, 0, s, halos, runs, nruns, g, o);
}

hipError_t launch_potential64(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                              const OutDesc& o, int px, hipStream_t s)
{
    switch (px) {
    case kPxSplit: launch_potential64_px<1, SUM_WAVES>(halos, runs, nruns, g, o, s); break;
    case kPxParts:
        if (parts_px(g, 1.0) == 1) launch_potential64_px<1, SUM_PARTS>(halos, runs, nruns, g, o, s);
        else launch_potential64_px<2, SUM_PARTS>(halos, runs, nruns, g, o, s);
        break;
    case 1: launch_potential64_px<1, SUM_PLAIN>(halos, runs, nruns, g, o, s); break;
    case 4: launch_potential64_px<4, SUM_PLAIN>(halos, runs, nruns, g, o, s); break;
    default: launch_potential64_px<2, SUM_PLAIN>(halos, runs, nruns, g, o, s); break;
    }
    return hipGetLastError();
}

}  // namespace lt
