// Arguments of the z sweep with the conserved update (mhd_sweep.hpp).
#pragma once
#include "mhd_launch.hpp"
#include "mhd_update.hpp"

namespace mhd {

struct SweepArgs {
    FluxSet<double> F;   // x and y fluxes (of z the count only)
    double* fz;          // where the z fluxes are left, or null
    double gm1;
    const double* tau_p;
    CCells s;            // the state the corrector starts from
    Cells so;            // and the one it writes
    const double *dx, *dy, *dz;
    int cells;           // along z, of one workgroup
};

// cells along z of a workgroup: runs of one length, at most kSweepTiles tiles of
// faces (16 tiles: 256^3 the same, 128^3 870 us for 859, 70 x 70 x 500 1.39 ms
// for 1.32, too few workgroups)
constexpr int kSweepTiles = 8;
inline int sweep_cells(const Dims& d) {
    const int most = kSweepTiles * kTileN - 1, runs = (d.nz0 + most - 1) / most;
    return (d.nz0 + runs - 1) / runs;
}
inline unsigned sweep_blocks(const Dims& d) {
    const int n = sweep_cells(d);
    return (unsigned)((d.nx0 + kTileX - 1) / kTileX) * d.ny0 * ((d.nz0 + n - 1) / n);
}

}  // namespace mhd

void launch_sweep_fp64(mhd_ctx* c, mhd::Src<double> s, const mhd::SweepArgs& a);
