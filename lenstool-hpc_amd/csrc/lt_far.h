// lt_far.h -- tile expansions of the halo sums (lt_far.hip): launcher and the rule that picks them.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "lt_device.h"
#include "lt_kernels.h"

namespace lt {

constexpr int kFarMaxHalos = 2048;   // halos of a model (the sets live in LDS)
constexpr int kFarMaxRuns = 16;      // runs of a model (every run is walked for every 16 x 16 block)

// What the far test reads of a halo (48 bytes, packed so that a wavefront's 64 are contiguous): its centre and the
// scaled frame in which a square of half side h is far when X^2 + Y^2 + f >= 36 h^2.
struct alignas(16) FarRec {
    double xh, yh;
    float a, b, c, d, f;
    float pad[3];
};
static_assert(sizeof(FarRec) == 48, "far record is 48 bytes");

void far_records(const HaloRec* recs, int nhalos, FarRec* out);

// What the rule looks at: of a model, the direct sum's cost; of a lens (a sample of it), how many times over the tiles that
// hold its halos are near to one halo, for tiles of half side 1: the mean area inside which a halo is near, by the
// area over which the halos lie. Taken to a quarter of an octave, so that samples of one model rarely differ in it.
struct FarStats {
    int nhalos = 0, nruns = 0;
    ModelCost cost;
};

FarStats far_stats(int nhalos, const std::vector<Run>& runs);
double halo_density(const HaloRec* recs, const std::vector<Run>& runs);

// How a map is summed: directly, or by tile expansions in work-groups of 64 (4 or 16 waves, or two of
// 8 or four of 4 for one root), 128 or 256 pixels a side.
enum class FarShape { Direct, Root64, Root64Wide, Root64Half, Root64Quarter, Root128, Root256 };

// The shape for a map of one lens. `whole`: the grid that the rows computed belong to (the grid itself, or the whole map where
// a part of it is computed on its own). *cost (may be NULL): estimated instructions per pixel of the form chosen.
FarShape far_shape(const FarStats& st, double density, int kind, int precision, const GridDesc& whole, double* cost);

// map o.kind of the grid in the shape that far_shape() gave (not Direct)
hipError_t launch_far(const HaloRec* halos, const FarRec* recs, const Run* runs, int nruns, int nhalos, const GridDesc& g,
                      const OutDesc& o, FarShape shape, hipStream_t s);

}  // namespace lt
