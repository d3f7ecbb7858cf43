// lt_kernels.h -- host-side declarations of the kernel launchers and of the model packer.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "lenstool_hip/lt_types.h"
#include "lt_device.h"

namespace lt {

// parts of a pixel's sum in the split form (lt_kernels64.hip), and the halos of an FP32C chunk (lt_kernels32.hip)
constexpr int kSplit = 8;
constexpr int kChunk32 = 8;

// px of a launch in the split form: a wave for each part of a row segment's halos, or the same sums by one wave
constexpr int kPxSplit = -1;
constexpr int kPxParts = -2;

// FP64 kernels (lt_kernels64.hip). px = pixels per thread (1, 2 or 4), kPxSplit or kPxParts; unit: every run's weight is 1.
hipError_t launch_hessian64(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                            const OutDesc& o, int px, bool unit, hipStream_t s);
hipError_t launch_gradient64(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                             const OutDesc& o, int px, hipStream_t s);
hipError_t launch_potential64(const HaloRec* halos, const Run* runs, int nruns, const GridDesc& g,
                              const OutDesc& o, int px, hipStream_t s);
// gradient at npts points for nsamples lens models (records of sample s start at s*halo_stride);
// outputs [nsamples*npts]
hipError_t launch_points_gradient64(const HaloRec* halos, const Run* runs, int nruns, const double* px,
                                   const double* py, int npts, int nsamples, int64_t halo_stride, double* gx,
                                   double* gy, hipStream_t s);
// map epilogue alone on device Hessian planes (kinds FIELDS, AMPLI, SHEAR, MASS)
hipError_t launch_epilogue64(const double* a, const double* b, const double* c, int64_t n, const OutDesc& o,
                             hipStream_t s);

// FP32-compensated kernels (lt_kernels32.hip).
hipError_t launch_hessian32(const HaloRec* halos64, const HaloRec32* halos32, const Run* runs, int nruns,
                            const GridDesc& g, const OutDesc& o, int px, bool unit, hipStream_t s);
// gradient / displacement maps; the model must be packed for gradient use (GradRec32 records)
hipError_t launch_gradient32(const HaloRec* halos64, const HaloRec32* recs32, const Run* runs, int nruns,
                             const GridDesc& g, const OutDesc& o, int px, hipStream_t s);

// potential maps; the model must be packed for potential use (PotRec32 records)
hipError_t launch_potential32(const HaloRec* halos64, const HaloRec32* recs32, const Run* runs, int nruns,
                              const GridDesc& g, const OutDesc& o, int px, hipStream_t s);

// Streaming device copy (16-byte vectors plus a byte tail).
hipError_t launch_copy(void* dst, const void* src, size_t bytes, hipStream_t s);
// x *= s on n doubles
hipError_t launch_scale(double* x, double s, size_t n, hipStream_t st);

// What a packed model is used for: the run split differs for the Kmap (runs also break on dlsds).
enum class Use { Gradient, Hessian, Kmap, Potential };

// Pack an SOA lens model into device records and runs. Returns an LT_* status; on error `err`
// names the offending halo.
int pack_model(const lt_potential_soa* lens, int nhalos, Use use, std::vector<HaloRec>& recs,
               std::vector<HaloRec32>& recs32, std::vector<Run>& runs, std::string& err);

// Instructions per pixel of the direct kernels, summed over a model's halos, by family (FAM_*): what the choices of
// launch shape go by.
enum : int { FAM_GRADIENT = 0, FAM_HESSIAN = 1, FAM_POTENTIAL = 2, FAM_TRACE = 3 };  // TRACE: xx + yy alone

struct ModelCost {
    double px[4] = {0, 0, 0, 0};
    // the split form's parts, in FP64 and in FP32C (where a part is whole chunks): which have halos, and over the runs how many
    int parts[2] = {0, 0};
    double nparts[2] = {0, 0};
};

int family_of(int kind);
ModelCost model_cost(const std::vector<Run>& runs);
double direct_cost(const ModelCost& c, int kind, int precision);

// Cosmology (lt_cosmo.cpp): angular distances in units of c/H0 and D_ls/D_s.
double cosmo_observer_object(double z, const lt_cosmo_param& c);
double cosmo_object_object(double z1, double z2, const lt_cosmo_param& c);

}  // namespace lt
